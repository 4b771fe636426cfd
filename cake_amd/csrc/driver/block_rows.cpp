// A run of Llama blocks over T > 1 rows, launched by one host call.
//
// The eight launches of a block take 594 us of GPU time in 9 blocks of width 2048 at 5 rows, and
// took 1118 us of wall time launched one by one from Python (14 us each: argument checks, views,
// allocations).  The caller checks and plans once per run, since every block has the same shapes;
// what is left per launch is the kernel library's own entry point (2 - 3 us).
//
// Of few rows the q/k/v, output and down products leave their sums in slabs, which the rotation and the next
// norm add up: six launches a block instead of up to eleven (a block of 8B at 45 rows 122 us, 116 so).
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
int cake_gemm_slabs(int dt, int kind, int cfg, int parts, const void* a, long long lda, const void* b,
                    long long ldb, float* ws, const void* zeros, int M, int N, int K, hipStream_t st);
int cake_slab_norm(int dt, const float* ws, int slabs, float* x, long long ldx, const void* bias, float alpha,
                   const void* w, int w32, float off, float eps, int ln, int M, int N, void* out, long long ldo,
                   hipStream_t st);
int cake_slab_rope(int dt, const float* ws, int slabs, void* q, int ldq, int T, int nh, int nkv, int hd,
                   const float* inv_freq, int pos0, int S, void* kc, void* vc, hipStream_t st);
}

namespace {

constexpr int kEpiStore = 0, kEpiResid32 = 1, kEpiSwiglu = 3;  // gemm_kernel.h

// of a product: rows form (0: none), else tile plan; slabs: as cake_gemm_slabs takes them
struct Form { int kind, cfg, splits, slabs; };

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
  float* slabs;                 // of the products that leave them
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
  // the product's slabs, their number (or minus an error)
  const auto slabs = [&](const Form& f, const void* a, const void* w, int N, int K) {
    return cake_gemm_slabs(r->dt, f.kind, f.cfg, f.splits, a, K, w, K, r->slabs, r->zeros, T, N, K, st);
  };
  // hidden += a w^T, and x = the norm of it by `ln` (null: none)
  const auto add_norm = [&](const Form& f, const void* a, const void* w, int K, const void* ln) {
    if (f.slabs) {
      const int n = slabs(f, a, w, H, K);
      return n < 0 ? -n : cake_slab_norm(r->dt, r->slabs, n, r->hidden, H, nullptr, 1.f, ln, 0, 0.f, r->eps, 0, T, H,
                                         r->x, H, st);
    }
    const int e = product(f, kEpiResid32, a, w, nullptr, H, K);
    return e || !ln ? e : cake_rmsnorm(r->dt, r->hidden, ln, r->eps, T, H, r->x, st);
  };
  uint16_t* q = static_cast<uint16_t*>(r->qkv);
  int e = r->n == 0 ? 0   // (one norm kernel at every place of the run)
          : r->down_form.slabs ? cake_slab_norm(r->dt, nullptr, 0, r->hidden, H, nullptr, 1.f, r->blocks[0].ln1, 0,
                                                0.f, r->eps, 0, T, H, r->x, H, st)
                               : cake_rmsnorm(r->dt, r->hidden, r->blocks[0].ln1, r->eps, T, H, r->x, st);
  for (int i = 0; !e && i < r->n; ++i) {
    const Block& b = r->blocks[i];
    if (r->qkv_form.slabs) {
      const int n = slabs(r->qkv_form, r->x, b.wqkv, nqkv, H);
      e = n < 0 ? -n : cake_slab_rope(r->dt, r->slabs, n, q, nqkv, T, r->nh, r->nkv, r->hd, r->inv_freq, r->pos0,
                                      r->S, b.kc, b.vc, st);
    } else {
      e = product(r->qkv_form, kEpiStore, r->x, b.wqkv, r->qkv, nqkv, H);
      if (!e)
        e = cake_rope_kv(r->dt, q, q + nq, q + nq + nk, nqkv, nqkv, T, r->nh, r->nkv, r->hd, r->inv_freq,
                         r->pos0, r->S, b.kc, b.vc, st);
    }
    if (!e)
      e = cake_flash_attn(r->dt, q, b.kc, b.vc, r->att, 1, r->nh, r->nkv, T, r->pos0 + T, r->hd,
                          strides, r->scale, 1, r->pos0, st);
    if (!e) e = add_norm(r->o_form, r->att, b.wo, nq, b.ln2);
    if (!e) e = product(r->gu_form, kEpiSwiglu, r->x, b.wgu, r->act, r->I, H);
    if (!e) e = add_norm(r->down_form, r->act, b.wd, r->I, i + 1 < r->n ? r->blocks[i + 1].ln1 : nullptr);
  }
  return e;
}
