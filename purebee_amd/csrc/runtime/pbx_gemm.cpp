// pbx_gemm.cpp -- launch path of the M >= 4 instruction: row scaling of the
// activations to fp16, the MFMA GEMM (pbx_gemm.hip) and, when the K blocks
// are split across workgroups, the reduction of the partial sums.  F32
// weights take the fp32 MFMA kernels, which read the activations as they are.

#include <algorithm>
#include <string>

#include "pbx_internal.h"

namespace {

struct GemmArgsHost {  // GemmArgs in pbx_gemm.hip
  const void *qs;
  const void *dsc;
  const void *X16;
  const void *X16lo;
  const float *inv;
  const float *bias;
  float *Y;
  int M, N, Npad, B, KS;
  int accumulate;
  const void *msc;
  int Mpad;
};

struct GemmF32ArgsHost {  // GemmF32Args in pbx_gemm.hip
  const void *W;
  const float *X;
  const float *bias;
  float *Y;
  int M, N, Npad, B, KS;
  int accumulate;
};

struct GemmRowsArgsHost {  // GemmRowsArgs in pbx_gemm.hip
  const void *qs;
  const void *dsc;
  const void *msc;
  const float *X;
  const float *bias;
  float *Y;
  int M, N, Npad, B;
  int accumulate;
};

const char *gemm_tag(int type) {
  switch (type) {
    case PBX_TYPE_Q4_0: return "q4";
    case PBX_TYPE_Q8_0: return "q8";
    case PBX_TYPE_Q4_1: return "q41";
    case PBX_TYPE_F16: return "f16";
    case PBX_TYPE_F32: return "f32";
    default: return nullptr;
  }
}

// `need` bytes of workspace: from ws when the caller brings one (an error if
// it is too small), else the context's grow-only GEMM buffer.
int workspace(pbx_ctx *c, const pbx_workspace *ws, size_t need, char **out) {
  if (ws) {
    if (!ws->ptr)
      return pbx_fail(c, PBX_ENOTSUP, "pbx_linear: no device workspace available");
    if (need > ws->bytes)
      return pbx_fail(c, PBX_EINVAL,
                      "pbx_linear: this shape needs %zu bytes of workspace, above the %zu-byte "
                      "limit of the no-allocation entry point",
                      need, ws->bytes);
    *out = (char *)ws->ptr;
    return PBX_OK;
  }
  int rc = pbx_ensure_dev(c, &c->d_gemm, &c->d_gemm_cap, need);
  if (rc) return rc;
  *out = (char *)c->d_gemm;
  return PBX_OK;
}

// Sum of the split-K partials into dY (+ bias, or accumulated).
int launch_reduce(pbx_ctx *c, float *part, const float *dBias, float *dY, int M, int N, int KS,
                  int accumulate, hipStream_t stream) {
  hipFunction_t fred = pbx_kernel_by_name(c, "pbx_gemm_reduce");
  if (!fred) return pbx_fail(c, PBX_ELOAD, "pbx_gemm: kernel pbx_gemm_reduce missing");
  int m = M, n = N, ks = KS, acc = accumulate;
  void *args[] = {&part, (void *)&dBias, &dY, &m, &n, &ks, &acc};
  const int64_t MN = (int64_t)M * N;
  return pbx_launch_fn(c, fred, "pbx_gemm_reduce", dim3((unsigned)((MN + 1023) / 1024)), dim3(256),
                       args, stream);
}

// F32 weights: fp32 MFMA.  M > 32: the LDS-DMA 128 x 128 kernel; otherwise
// wave tile 16*MT x 16*NT (MT 1 / 2 for M <= 16 / <= 32), K split for about
// eight waves per CU.
int launch_f32(pbx_ctx *c, const pbx_weight *w, const float *dX, int M, const float *dBias,
               float *dY, int accumulate, hipStream_t stream, const pbx_workspace *ws) {
  const int N = (int)w->N, B = (int)w->B;
  if (M > 32) {
    // 128 x 128 tiles on the LDS-DMA kernel, K split (16-k steps) for about
    // one workgroup per CU
    const int nwg = (N + 127) / 128, mtiles = (M + 127) / 128, wgs = nwg * mtiles;
    int KS = 1;
    if (wgs < c->cu_count) KS = std::min({2 * B, 8, (c->cu_count + wgs - 1) / wgs});
    float *part = nullptr;
    if (KS > 1) {
      char *p = nullptr;
      int rc = workspace(c, ws, (size_t)KS * M * N * 4, &p);
      if (rc) return rc;
      part = (float *)p;
    }
    hipFunction_t fg = pbx_kernel_by_name(c, "pbx_gemm_f32_big");
    if (!fg) return pbx_fail(c, PBX_ELOAD, "pbx_gemm: kernel pbx_gemm_f32_big missing");
    GemmF32ArgsHost g{w->qs, dX, KS == 1 ? dBias : nullptr, KS == 1 ? dY : part,
                      M, N, (int)w->Npad, B, KS, KS == 1 ? accumulate : 0};
    void *args[] = {&g};
    int rc = pbx_launch_fn(c, fg, "pbx_gemm_f32_big", dim3(nwg, mtiles, KS), dim3(256), args, stream);
    if (rc || KS == 1) return rc;
    return launch_reduce(c, part, dBias, dY, M, N, KS, accumulate, stream);
  }
  const int MT = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const int mtiles = (M + 16 * MT - 1) / (16 * MT);
  int NT;
  if (MT == 1)
    NT = ((N + 255) / 256) * mtiles >= 2 * c->cu_count ? 4
         : ((N + 127) / 128) * mtiles >= 2 * c->cu_count ? 2 : 1;
  else
    NT = MT == 2 ? 2 : 4;
  const int nwg = (N + 64 * NT - 1) / (64 * NT);
  int KS = 1;
  const int waves = nwg * mtiles * 4;
  if (waves < 8 * c->cu_count) KS = std::min({B, 8, (8 * c->cu_count + waves - 1) / waves});
  float *part = nullptr;
  if (KS > 1) {
    char *p = nullptr;
    int rc = workspace(c, ws, (size_t)KS * M * N * 4, &p);
    if (rc) return rc;
    part = (float *)p;
  }
  const std::string name = "pbx_gemm_f32_m" + std::to_string(MT) + "_n" + std::to_string(NT);
  hipFunction_t fg = pbx_kernel_by_name(c, name);
  if (!fg) return pbx_fail(c, PBX_ELOAD, "pbx_gemm: kernel %s missing", name.c_str());
  GemmF32ArgsHost g{w->qs, dX, KS == 1 ? dBias : nullptr, KS == 1 ? dY : part,
                    M, N, (int)w->Npad, B, KS, KS == 1 ? accumulate : 0};
  void *args[] = {&g};
  int rc = pbx_launch_fn(c, fg, name.c_str(), dim3(nwg, mtiles, KS), dim3(256), args, stream);
  if (rc || KS == 1) return rc;
  return launch_reduce(c, part, dBias, dY, M, N, KS, accumulate, stream);
}

// Few activation rows, one launch: 16 * MT rows of X and 16 * NT rows of W a
// workgroup.
int launch_rows(pbx_ctx *c, const pbx_weight *w, const float *dX, int M, const float *dBias,
                float *dY, int accumulate, hipStream_t stream) {
  const int N = (int)w->N, B = (int)w->B, chunks = (B + 7) / 8;
  // Every workgroup loads and splits its activations, so the widest tile wins
  // that still gives three quarters of the CUs a workgroup: 8192 x 2048 at 16
  // rows 12.0 us with NT = 2 (256 workgroups) against 15.0 with NT = 1; 2048 x
  // 8192 at 32 rows 28 us in 16 x 16 tiles (256) against 37 and 43 in 16 x 32
  // and 32 x 16; 3072 x 2048 at 32 rows 12.0 in 16 x 32 (192) against 14.7.
  auto wgs = [&](int mt, int nt) {
    return (int64_t)((N + 16 * nt - 1) / (16 * nt)) * ((M + 16 * mt - 1) / (16 * mt));
  };
  const int64_t enough = c->cu_count * 3 / 4;
  int MT = 1, NT = 1;
  if (M > 16 && wgs(2, 2) >= enough) MT = NT = 2;
  else if (M <= 16 && wgs(1, 4) >= enough) NT = 4;
  else if (wgs(1, 2) >= enough) NT = 2;
  // More than one round of workgroups: those of one a CU walk the tiles with
  // the activations in registers (K <= 2048).  16384 x 2048 Q8_0 at 20 rows
  // 21.6 us against 28.6; 128256 x 2048 Q6_K at 5 rows 72 against 98
  // (in turn on one box; 80 on others).
  const bool loop = chunks <= 8 && NT > 1 && wgs(MT, NT) >= 2 * c->cu_count;
  if (loop) NT = MT == 1 ? 2 : 1;
  const std::string name = std::string("pbx_gemm_rows_") +
                           (w->type == PBX_TYPE_Q6_K ? "q6k" : gemm_tag(w->type)) + "_m" +
                           std::to_string(MT) + "_n" + std::to_string(NT) + (loop ? "l" : "");
  hipFunction_t f = pbx_kernel_by_name(c, name);
  if (!f) return pbx_fail(c, PBX_ELOAD, "pbx_gemm: kernel %s missing", name.c_str());
  const int tiles = (N + 16 * NT - 1) / (16 * NT), mtiles = (M + 16 * MT - 1) / (16 * MT);
  GemmRowsArgsHost g{w->qs, w->d, w->m, dX, dBias, dY, M, N, (int)w->Npad, B, accumulate};
  void *args[] = {&g};
  return pbx_launch_fn(c, f, name.c_str(),
                       dim3(loop ? std::min(tiles, std::max(1, c->cu_count / mtiles)) : tiles, mtiles),
                       dim3(64 * std::min(8, chunks)), args, stream);
}

// Up to PBX_GEMM_ROWS_M rows, where the one-launch kernel loses because every
// workgroup converts its rows' whole K (about 3.2 us a 1024 columns of 16
// rows, however few the workgroups):
// * few columns and long rows: pbx_gemm_<type>_p16, K split over workgroups.
//   Q4_0 2048 x 8192: 16 rows 18.5 us against 27.3, 12 rows 18.3 / 23.3, 8 rows
//   18.2 / 20.5; 2048 x 6144, 11 rows 15.7 / 18.6; 2048 x 4096, 16 rows 12.9 /
//   15.4; so from 64 K activation values on.  Q4_1, whose block sums cost the
//   one-launch kernel more, from 48 K (2048 x 8192, 8 rows 19.7 / 24.0).  Not
//   for 4 rows (F16 2048 x 16384 33 / 30), nor past half the CUs' tiles.
bool few_columns(const pbx_ctx *c, const pbx_weight *w, int M) {
  const int64_t values = (int64_t)M * w->B * 32;
  return M > 4 && M <= 16 && (w->N + 15) / 16 <= c->cu_count / 2 &&
         values >= (w->type == PBX_TYPE_Q4_1 ? 48 << 10 : 64 << 10);
}
// * many rounds of 32 x 32 tiles of more than 2048 columns (shorter rows stay
//   in registers over the rounds): the prepared LDS-DMA GEMM.  Q4_0 32 rows
//   16384 x 4096 50.4 us against 57.1, 32768 x 2304 48 / 68, 32768 x 8192 170 /
//   210; 20 rows 16384 x 8192 90 / 88, 32768 x 4096 80 / 90; 32 rows 16384 x
//   2304 35.1 / 34.6, Q8_0 38 / 34.5.  A weight beyond
//   the 256 MB of the last-level cache comes from HBM either way, and the
//   one-launch kernel streams it better (F16 32768 x 8192, 32 rows 248 / 206).
bool many_columns(const pbx_ctx *c, const pbx_weight *w, int M) {
  const int64_t tiles = (w->N + 31) / 32;
  return M > 16 && w->B > 64 && M * tiles >= 64 * (int64_t)c->cu_count &&
         M * tiles * w->B >= 5120 * (int64_t)c->cu_count &&
         w->N * pbx_type_row_bytes(w->type, w->K) <= 256 << 20;
}

// Workspace of the prepared GEMM: the fp16 pair, the row scales and the
// split-K partials.
struct GemmSpace {
  size_t x16, inv, part;
  size_t total() const { return 2 * x16 + inv + part; }
};
GemmSpace gemm_space(const pbx_gemm_plan &p, int N, int K) {
  return {((size_t)p.Mpad * K * 2 + 255) / 256 * 256, ((size_t)p.Mpad * 4 + 255) / 256 * 256,
          p.KS > 1 ? (size_t)p.KS * p.M * N * 4 : 0};
}

}  // namespace

int pbx_gemm_make_plan(pbx_ctx *c, const pbx_weight *w, int M, pbx_gemm_plan *p, bool swiglu) {
  if (!gemm_tag(w->type) || w->type == PBX_TYPE_F32)
    return pbx_fail(c, PBX_ENOTSUP, "pbx_gemm: weight type %d has no fp16 MFMA path", w->type);
  if (M <= 0 || M > 65535) return pbx_fail(c, PBX_ENOTSUP, "pbx_gemm: M=%d out of range", M);
  const int N = (int)w->N, B = (int)w->B;
  const int Mpad = (M + 127) / 128 * 128, mtiles = Mpad / 128, nwg = (N + 127) / 128;
  int KS = 1;
  int mt_rows = 128;
  int mtl = mtiles;
  // 128 x 128 tiles where they give two workgroups a CU (the prefill's
  // gate|up): 16384 x 2048 at 2000 rows 312 us against 337 in 64-row tiles
  // (half the outputs for the same codes unpacked).  Otherwise
  // 64-row M tiles (pbx_gemm_<type>_b64) with the K split to two workgroups
  // a CU (PBX_GEMM_M64 = workgroups a CU, 0: the 128-row tiles at about one
  // a CU): 8192 x 2048 at 512 rows 57.7 against 63.1 us in 128-row tiles at
  // one a CU, 3072 x 2048 at 2000 80 against 86.
  const int wgs = nwg * mtiles;
  const char *e = getenv("PBX_GEMM_M64");
  const int per_cu = e ? atoi(e) : 2;
  if (per_cu > 0 && wgs < per_cu * c->cu_count) {
    mt_rows = 64;
    mtl = Mpad / 64;
    const int w64 = nwg * mtl;
    if (w64 < per_cu * c->cu_count)
      KS = std::min({B, 8, (per_cu * c->cu_count + w64 - 1) / w64});
  } else if (wgs < c->cu_count) {
    KS = std::min({B, 8, (c->cu_count + wgs - 1) / wgs});
  }
  p->M = M;
  p->Mpad = Mpad;
  p->mtiles = mtl;
  p->nwg = nwg;
  p->KS = KS;
  // gate|up with silu(gate) * up in the epilogue (no K split, 64
  // hidden columns a workgroup, 32-bit weight offsets);
  // PBX_GEMM_SWIGLU=0 keeps gate and up side by side
  const char *sw_env = getenv("PBX_GEMM_SWIGLU");
  p->swiglu = swiglu && KS == 1 && N % 128 == 0 &&
              (double)N * pbx_type_row_bytes(w->type, w->K) < 4294967296.0 &&
              !(sw_env && sw_env[0] == '0');
  p->name = std::string("pbx_gemm_") + gemm_tag(w->type) +
            (mt_rows == 64 ? "_b64" : "_big") + (p->swiglu ? "_sw" : "");
  return PBX_OK;
}

int pbx_gemm_run(pbx_ctx *c, const pbx_weight *w, const pbx_gemm_plan &p, const void *x16,
                 const void *x16lo, const float *inv, const float *dBias, float *out,
                 int accumulate, hipStream_t stream) {
  hipFunction_t fg = pbx_kernel_by_name(c, p.name);
  if (!fg) return pbx_fail(c, PBX_ELOAD, "pbx_gemm: kernel %s missing", p.name.c_str());
  GemmArgsHost g{w->qs, w->d, x16, x16lo, inv, p.KS == 1 ? dBias : nullptr, out,
                 p.M, (int)w->N, (int)w->Npad, (int)w->B, p.KS, p.KS == 1 ? accumulate : 0, w->m, p.Mpad};
  void *args[] = {&g};
  return pbx_launch_fn(c, fg, p.name.c_str(), dim3(p.nwg, p.mtiles, p.KS), dim3(256), args, stream);
}

int pbx_gemm_launch(pbx_ctx *c, const pbx_weight *w, const float *dX, int64_t M64,
                    const float *dBias, float *dY, int accumulate, hipStream_t stream,
                    const pbx_workspace *wsp) {
  if (!gemm_tag(w->type) && w->type != PBX_TYPE_Q6_K)
    return pbx_fail(c, PBX_ENOTSUP, "pbx_gemm: weight type %d has no MFMA path", w->type);
  if (M64 > 65535) return pbx_fail(c, PBX_ENOTSUP, "pbx_gemm: M=%lld too large", (long long)M64);
  if (w->type == PBX_TYPE_F32)
    return launch_f32(c, w, dX, (int)M64, dBias, dY, accumulate, stream, wsp);
  if (w->type == PBX_TYPE_Q6_K) {
    if (w->B > 512)
      return pbx_fail(c, PBX_ENOTSUP, "pbx_linear: K=%lld exceeds the Q6_K limit of 16384",
                      (long long)w->K);
    return launch_rows(c, w, dX, (int)M64, dBias, dY, accumulate, stream);
  }
  const int M = (int)M64, N = (int)w->N, K = (int)w->B * 32;
  pbx_gemm_plan p;
  int rc;
  if (few_columns(c, w, M)) {
    p.M = M;
    p.Mpad = 16;
    p.mtiles = 1;
    p.nwg = (N + 63) / 64;
    p.KS = 8;  // the tiles alone are a wave each for at most half of the CUs
    p.name = std::string("pbx_gemm_") + gemm_tag(w->type) + "_p16";
  } else if ((M > PBX_GEMM_ROWS_M || many_columns(c, w, M)) &&
             (rc = pbx_gemm_make_plan(c, w, M, &p))) {
    return rc;
  }
  if (!p.M) {
    // One launch on the fp32 rows: no workspace is used.  A caller that brings
    // one is still refused a K whose fp16 pair it could not hold: its limit
    // does not depend on the kernel that a shape takes.
    char *unused = nullptr;
    const size_t pair = (size_t)(M <= 16 ? 16 : 32) * K * 4;
    rc = wsp ? workspace(c, wsp, pair, &unused) : PBX_OK;
    return rc ? rc : launch_rows(c, w, dX, M, dBias, dY, accumulate, stream);
  }
  const GemmSpace sp = gemm_space(p, N, K);
  char *ws = nullptr;
  if ((rc = workspace(c, wsp, sp.total(), &ws))) return rc;
  // fp16 activations and their fp16 rounding residuals
  void *x16 = ws;
  void *x16lo = ws + sp.x16;
  float *inv = (float *)(ws + 2 * sp.x16);
  float *part = (float *)(ws + 2 * sp.x16 + sp.inv);
  hipFunction_t fprep = pbx_kernel_by_name(c, "pbx_gemm_prep_x");
  if (!fprep) return pbx_fail(c, PBX_ELOAD, "pbx_gemm: kernel pbx_gemm_prep_x missing");
  {
    int m = M, k = K;
    void *args[] = {(void *)&dX, &x16, &x16lo, &inv, &m, &k};
    if ((rc = pbx_launch_fn(c, fprep, "pbx_gemm_prep_x", dim3(p.Mpad), dim3(256), args, stream)))
      return rc;
  }
  if ((rc = pbx_gemm_run(c, w, p, x16, x16lo, inv, dBias, p.KS == 1 ? dY : part, accumulate,
                         stream)))
    return rc;
  if (p.KS > 1) return launch_reduce(c, part, dBias, dY, M, N, p.KS, accumulate, stream);
  return PBX_OK;
}

int pbx_gemm_enqueue(pbx_ctx *c, const pbx_weight *w, const float *dX, int64_t M,
                     const float *dBias, float *dY, hipStream_t stream, const pbx_workspace *ws) {
  return pbx_gemm_launch(c, w, dX, M, dBias, dY, 0, stream, ws);
}
