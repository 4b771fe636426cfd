// A run of Llama blocks over T > 1 rows, launched by one host call.
//
// The eight launches of a block take 594 us of GPU time in 9 blocks of width 2048 at 5 rows, and
// took 1118 us of wall time launched one by one from Python (14 us each: argument checks, views,
// allocations).  The caller checks and plans once per run, since every block has the same shapes;
// what is left per launch is the kernel library's own entry point (2 - 3 us).
#include <hip/hip_runtime.h>
#include <stdint.h>

#define CAKE_API extern "C" __attribute__((visibility("default")))

extern "C" {
int cake_rmsnorm(int dt, const float* x, const void* w, float eps, int T, int H, void* out,
                 hipStream_t st);
int cake_rope_kv(int dt, void* q, const void* k, const void* v, int ldq, int ld, int T, int nh,
                 int nkv, int hd, const float* inv_freq, int pos0, int S, void* kc, void* vc,
                 hipStream_t st);
int cake_flash_attn(int dt, const void* q, const void* k, const void* v, void* o, int B, int H,
                    int Hkv, int N, int M, int D, const long long* strides, float scale,
                    int causal, int pos0, hipStream_t st);
int cake_gemm_rows(int dt, int epi, int kind, const void* a, long long lda, const void* b,
                   long long ldb, void* c, long long ldc, const void* bias, void* resid,
                   long long ldr, float* ws, void* tick, const void* zeros, int M, int N, int K,
                   float alpha, hipStream_t st);
int cake_gemm_scaled(int dt, int epi, int cfg, int splits, const void* a, long long lda,
                     const void* b, long long ldb, void* c, long long ldc, const void* bias,
                     void* resid, long long ldr, float* ws, void* tick, const void* zeros, int M,
                     int N, int K, float alpha, hipStream_t st);
}

namespace {

constexpr int kEpiStore = 0, kEpiResid32 = 1, kEpiSwiglu = 3;  // gemm_kernel.h

struct Form { int kind, cfg, splits; };  // of a product: rows form (0: none), else tile plan

struct Block {  // device pointers of one block; the cache rows [nkv][S][hd] are this block's own
  const void *ln1, *wqkv, *wo, *ln2, *wgu, *wd;
  void *kc, *vc;
};

}  // namespace

// (mirrored by ops/llama_rows.py)
struct CakeBlockRun {
  const Block* blocks;
  float* hidden;                // [T][H] f32, in place
  void *x, *qkv, *att, *act;    // [T][H], [T][(nh + 2 nkv) hd], [T][nh hd], [T][I]
  const float* inv_freq;
  const void* zeros;
  float* ws;                    // split-k slabs of the tile plans
  float* rows_ws;               // workspace of the stream form
  void* tick;                   // counters of either
  Form qkv_form, o_form, gu_form, down_form;
  int n, dt, T, H, I, nh, nkv, hd, S, pos0;
  float eps, scale;
};

// 0, or the HIP error of the first launch that failed (the blocks behind it are not launched)
CAKE_API int cake_block_rows(const CakeBlockRun* r, hipStream_t st) {
  if (!r || r->n < 0 || r->T < 1 || r->pos0 < 0 || r->pos0 + r->T > r->S)
    return (int)hipErrorInvalidValue;
  const int T = r->T, H = r->H, nq = r->nh * r->hd, nk = r->nkv * r->hd, nqkv = nq + 2 * nk;
  const long long Sh = (long long)r->S * r->hd;
  // [batch, head, row] strides of q (a column block of qkv), the cache twice, the output
  const long long strides[12] = {(long long)T * nqkv, r->hd, nqkv, r->nkv * Sh, Sh, r->hd,
                                 r->nkv * Sh, Sh, r->hd, (long long)T * nq, r->hd, nq};
  const auto product = [&](const Form& f, int epi, const void* a, const void* w, void* c, int N,
                           int K) {
    void* resid = epi == kEpiResid32 ? r->hidden : nullptr;
    const long long ldr = resid ? N : 0, ldc = resid ? 0 : N;
    return f.kind ? cake_gemm_rows(r->dt, epi, f.kind, a, K, w, K, c, ldc, nullptr, resid, ldr,
                                   r->rows_ws, r->tick, r->zeros, T, N, K, 1.f, st)
                  : cake_gemm_scaled(r->dt, epi, f.cfg, f.splits, a, K, w, K, c, ldc, nullptr,
                                     resid, ldr, f.splits > 1 ? r->ws : nullptr, r->tick, r->zeros, T,
                                     N, K, 1.f, st);
  };
  uint16_t* q = static_cast<uint16_t*>(r->qkv);
  for (int i = 0; i < r->n; ++i) {
    const Block& b = r->blocks[i];
    int e = cake_rmsnorm(r->dt, r->hidden, b.ln1, r->eps, T, H, r->x, st);
    if (!e) e = product(r->qkv_form, kEpiStore, r->x, b.wqkv, r->qkv, nqkv, H);
    if (!e)
      e = cake_rope_kv(r->dt, q, q + nq, q + nq + nk, nqkv, nqkv, T, r->nh, r->nkv, r->hd,
                       r->inv_freq, r->pos0, r->S, b.kc, b.vc, st);
    if (!e)
      e = cake_flash_attn(r->dt, q, b.kc, b.vc, r->att, 1, r->nh, r->nkv, T, r->pos0 + T, r->hd,
                          strides, r->scale, 1, r->pos0, st);
    if (!e) e = product(r->o_form, kEpiResid32, r->att, b.wo, nullptr, H, nq);
    if (!e) e = cake_rmsnorm(r->dt, r->hidden, b.ln2, r->eps, T, H, r->x, st);
    if (!e) e = product(r->gu_form, kEpiSwiglu, r->x, b.wgu, r->act, r->I, H);
    if (!e) e = product(r->down_form, kEpiResid32, r->act, b.wd, nullptr, H, r->I);
    if (e) return e;
  }
  return 0;
}
