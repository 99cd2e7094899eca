// Typed entry points for KDA: the chunked forward (kda_intra + kda_state) and
// the token-by-token recurrent form (kda_recurrent).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "runtime.h"

using namespace tmhip;

namespace {

constexpr int kChunk = 64, kKeyDim = 128, kValueDim = 128;
constexpr size_t kChunkBytes = 74240;  // workspace bytes per (head, chunk)

// Kernel argument block; must match struct KdaParams in kda.hip.
struct KdaParams {
  const void* q;
  const void* k;
  const void* v;
  const float* g;
  const void* beta;
  const float* s0;
  void* o;
  float* st;
  void* ws;
  int B, T, H, NC;
  int c0, c1;
  float scale;
  int beta_bf16;
};

Kernel& intra_kernel() {
  static Kernel k("kda_intra");
  return k;
}
Kernel& state_kernel() {
  static Kernel k("kda_state");
  return k;
}
Kernel& recurrent_kernel() {
  static Kernel k("kda_recurrent");
  return k;
}
Kernel& recurrent_v4_kernel() {
  static Kernel k("kda_recurrent_v4");
  return k;
}

// Chunks of each (batch, head) that go through the two kernels before the next
// ones take their place in the workspace.  kda_intra writes the workspace and
// kda_state reads it back, which the 256 MB Infinity Cache serves while the
// chunks of one place fit; every segment costs two launches and the ends of two
// grids.  A workspace that several calls share (the caller's): 3072 chunks (228 MB).
// One workspace per plan (compact): the calls of other plans evict each other's,
// so segments of at most 1700 chunks (126 MB), from 2000 on.  us with 1 / 2 / 3 / 4
// segments, shared, and with three plans' own workspaces in turn:
//   B = 1 T = 6200  H = 16 (1552 chunks) 137 / 151 / 171 / 179, 142 / 151 / 170 / 177
//   B = 1 T = 8192  H = 16 (2048) 170 / 180 / 207 / 201, 236 / 182 / 208 / 201
//   B = 2 T = 4096  H = 24 (3072) 214 / 222 / 252 / 267, 243 / 222 / 253 / 267
//   B = 1 T = 14000 H = 16 (3504) 380 / 293 / 317 / 328, 400 / 326 / 316 / 329
//   B = 1 T = 16384 H = 16 (4096) 476 / 341 / 368 / 364, 482 / 416 / 367 / 363
//   B = 4 T = 8192  H = 16 (8192) 661 / 688 / 499 / 522, 661 / 690 / 540 / 553
// Segments of fewer than 4 chunks would mostly hand states over (16 sequences of
// 1024, H = 32: 4 chunks 598 of 665, 2 chunks 755): then one pass.
int segment_chunks(long long bh, long long nc, bool compact) {
  const long long most = compact && bh * nc > 2000 ? 1700 : 3072;
  if (bh * nc <= most || most / bh < 4) return (int)nc;
  const long long nseg = (nc + most / bh - 1) / (most / bh);
  return (int)((nc + nseg - 1) / nseg);
}

}  // namespace

extern "C" size_t tm_kda_workspace_size(int batch, int seq_len, int heads, int key_dim,
                                        int value_dim, int chunk_size) {
  if (batch < 0 || seq_len < 0 || heads < 0 || key_dim != kKeyDim || value_dim != kValueDim ||
      chunk_size != kChunk)
    return 0;
  const size_t nc = ((size_t)seq_len + kChunk - 1) / kChunk;
  return (size_t)batch * heads * nc * kChunkBytes;
}

extern "C" size_t tm_kda_compact_workspace_size(int batch, int seq_len, int heads, int key_dim,
                                                int value_dim, int chunk_size) {
  const size_t all = tm_kda_workspace_size(batch, seq_len, heads, key_dim, value_dim, chunk_size);
  if (all == 0) return 0;
  const long long bh = (long long)batch * heads, nc = ((long long)seq_len + kChunk - 1) / kChunk;
  const int seg = segment_chunks(bh, nc, true);
  // the place of one segment and, behind it, the state handed to the next
  return seg >= nc ? all
                   : (size_t)bh * (seg * kChunkBytes + kKeyDim * kValueDim * sizeof(float));
}

// Both entry points.
static int kda_chunk_fwd(const char* op, bool compact, const void* q, const void* k, const void* v,
                         const float* g, const void* beta, const float* initial_state, void* o,
                         float* final_state, int batch, int seq_len, int heads, int key_dim,
                         int value_dim, int chunk_size, float scale, int beta_dtype,
                         void* workspace, size_t workspace_bytes, void* stream) {
  if (batch < 0 || seq_len < 0 || heads < 0 || key_dim <= 0 || value_dim <= 0 || chunk_size <= 0)
    return fail(TM_ERR_INVALID_ARG, "%s: B=%d T=%d H=%d Dk=%d Dv=%d chunk=%d",
                op, batch, seq_len, heads, key_dim, value_dim, chunk_size);
  if (key_dim != kKeyDim || value_dim != kValueDim || chunk_size != kChunk)
    return fail(TM_ERR_UNSUPPORTED,
                "%s: key_dim=%d value_dim=%d chunk_size=%d (supported: 128, 128, 64)",
                op, key_dim, value_dim, chunk_size);
  if (beta_dtype != TM_DT_F32 && beta_dtype != TM_DT_BF16)
    return fail(TM_ERR_INVALID_ARG, "%s: beta_dtype %d", op, beta_dtype);
  if (!std::isfinite(scale)) return fail(TM_ERR_INVALID_ARG, "%s: scale", op);
  if (batch == 0 || heads == 0) return 0;
  if (seq_len > 0 && (!q || !k || !v || !g || !beta || !o))
    return fail(TM_ERR_INVALID_ARG, "%s: null buffer", op);
  const size_t need =
      compact
          ? tm_kda_compact_workspace_size(batch, seq_len, heads, key_dim, value_dim, chunk_size)
          : tm_kda_workspace_size(batch, seq_len, heads, key_dim, value_dim, chunk_size);
  if (need > 0 && (!workspace || workspace_bytes < need))
    return fail(TM_ERR_INVALID_ARG, "%s: workspace of %zu bytes, need %zu", op,
                workspace_bytes, need);
  if (seq_len == 0 && !final_state) return 0;
  for (const void* ptr : {q, k, v, (const void*)g, (const void*)o, (const void*)workspace})
    if (ptr && !aligned16(ptr))
      return fail(TM_ERR_INVALID_ARG, "%s: buffers must be 16-byte aligned", op);
  if ((initial_state && !aligned16(initial_state)) || (final_state && !aligned16(final_state)))
    return fail(TM_ERR_INVALID_ARG, "%s: state buffers must be 16-byte aligned", op);
  const long long nc = ((long long)seq_len + kChunk - 1) / kChunk;
  const long long bh = (long long)batch * heads;
  if (bh * nc > 0x7fffffffLL || (long long)batch * seq_len * heads > 0x7fffffffLL)
    return fail(TM_ERR_UNSUPPORTED, "%s: problem too large for 32-bit indexing", op);
  if (!api()) return TM_ERR_NO_RUNTIME;
  clear_error();

  KdaParams p;
  memset(&p, 0, sizeof p);
  p.q = q; p.k = k; p.v = v; p.g = g; p.beta = beta;
  p.s0 = initial_state; p.o = o; p.st = final_state; p.ws = workspace;
  p.B = batch; p.T = seq_len; p.H = heads; p.NC = (int)nc;
  p.scale = scale;
  p.beta_bf16 = beta_dtype == TM_DT_BF16 ? 1 : 0;

  const int seg = segment_chunks(bh, nc, compact);
  float* hand = (float*)((char*)workspace + (size_t)bh * seg * kChunkBytes);
  p.NC = seg;
  for (int c0 = 0;; c0 += seg) {
    p.c0 = c0;
    p.c1 = (int)std::min<long long>(nc, c0 + seg);
    p.st = p.c1 < nc ? hand : final_state;
    if (p.c1 > c0) {
      // two workgroups per CU (their LDS and registers admit no third), each
      // walking its share of the chunks
      const long long grid = std::min<long long>(bh * (p.c1 - c0), 2LL * cu_count());
      const int rc = launch(intra_kernel(), dim3((unsigned)grid), dim3(256), 0, stream, p);
      if (rc) return rc;
    }
    const int rc = launch(state_kernel(), dim3((unsigned)(bh * (kValueDim / 16))), dim3(192), 0,
                          stream, p);
    if (rc || p.c1 >= nc) return rc;
    p.s0 = hand;
  }
}

extern "C" int tm_kda_chunk_fwd(const void* q, const void* k, const void* v, const float* g,
                                const void* beta, const float* initial_state, void* o,
                                float* final_state, int batch, int seq_len, int heads,
                                int key_dim, int value_dim, int chunk_size, float scale,
                                int beta_dtype, void* workspace, size_t workspace_bytes,
                                void* stream) {
  return kda_chunk_fwd("tm_kda_chunk_fwd", false, q, k, v, g, beta, initial_state, o, final_state,
                       batch, seq_len, heads, key_dim, value_dim, chunk_size, scale, beta_dtype,
                       workspace, workspace_bytes, stream);
}

extern "C" int tm_kda_chunk_fwd_compact(const void* q, const void* k, const void* v,
                                        const float* g, const void* beta,
                                        const float* initial_state, void* o, float* final_state,
                                        int batch, int seq_len, int heads, int key_dim,
                                        int value_dim, int chunk_size, float scale,
                                        int beta_dtype, void* workspace, size_t workspace_bytes,
                                        void* stream) {
  return kda_chunk_fwd("tm_kda_chunk_fwd_compact", true, q, k, v, g, beta, initial_state, o,
                       final_state, batch, seq_len, heads, key_dim, value_dim, chunk_size, scale,
                       beta_dtype, workspace, workspace_bytes, stream);
}

extern "C" int tm_kda_recurrent_fwd(const void* q, const void* k, const void* v, const float* g,
                                    const void* beta, const float* initial_state, void* o,
                                    float* final_state, int batch, int seq_len, int heads,
                                    int key_dim, int value_dim, float scale, int beta_dtype,
                                    void* stream) {
  if (batch < 0 || seq_len < 0 || heads < 0 || key_dim <= 0 || value_dim <= 0)
    return fail(TM_ERR_INVALID_ARG, "tm_kda_recurrent_fwd: B=%d T=%d H=%d Dk=%d Dv=%d", batch,
                seq_len, heads, key_dim, value_dim);
  if (key_dim != kKeyDim || value_dim != kValueDim)
    return fail(TM_ERR_UNSUPPORTED,
                "tm_kda_recurrent_fwd: key_dim=%d value_dim=%d (supported: 128, 128)", key_dim,
                value_dim);
  if (beta_dtype != TM_DT_F32 && beta_dtype != TM_DT_BF16)
    return fail(TM_ERR_INVALID_ARG, "tm_kda_recurrent_fwd: beta_dtype %d", beta_dtype);
  if (!std::isfinite(scale)) return fail(TM_ERR_INVALID_ARG, "tm_kda_recurrent_fwd: scale");
  if (batch == 0 || heads == 0) return 0;
  if (seq_len > 0 && (!q || !k || !v || !g || !beta || !o))
    return fail(TM_ERR_INVALID_ARG, "tm_kda_recurrent_fwd: null buffer");
  if (seq_len == 0 && !final_state) return 0;
  for (const void* ptr : {q, k, v, (const void*)g})
    if (ptr && !aligned16(ptr))
      return fail(TM_ERR_INVALID_ARG, "tm_kda_recurrent_fwd: q, k, v, g must be 16-byte aligned");
  if ((long long)batch * seq_len * heads * kKeyDim > 0x7fffffffffffLL ||
      (long long)batch * heads * (kValueDim / 16) > 0x7fffffffLL)
    return fail(TM_ERR_UNSUPPORTED, "tm_kda_recurrent_fwd: problem too large");
  if (!api()) return TM_ERR_NO_RUNTIME;
  clear_error();
  KdaParams p;
  memset(&p, 0, sizeof p);
  p.q = q; p.k = k; p.v = v; p.g = g; p.beta = beta;
  p.s0 = initial_state; p.o = o; p.st = final_state;
  p.B = batch; p.T = seq_len; p.H = heads;
  p.scale = scale;
  p.beta_bf16 = beta_dtype == TM_DT_BF16 ? 1 : 0;
  // one wave per (head, 16 value columns), or per (head, 32 value columns)
  // with 16-byte state accesses when both state buffers (or null) are 16-byte
  // aligned
  const bool v4 = ((reinterpret_cast<uintptr_t>(initial_state) |
                    reinterpret_cast<uintptr_t>(final_state)) & 15) == 0;
  const long long waves = (long long)batch * heads * (kValueDim / (v4 ? 32 : 16));
  return launch(v4 ? recurrent_v4_kernel() : recurrent_kernel(), dim3((unsigned)waves), dim3(64),
                0, stream, p);
}
