// A run of Llama blocks over T > 1 rows, launched by one host call.
//
// The eight launches of a block take 594 us of GPU time in 9 blocks of width 2048 at 5 rows, and
// took 1118 us of wall time launched one by one from Python (14 us each: argument checks, views,
// allocations).  The caller checks and plans once per run, since every block has the same shapes;
// what is left per launch is the kernel library's own entry point (2 - 3 us).
//
// Where the caller reads the last rows of the result only (a prompt's logits), the last block computes keys and
// values of all rows, and what follows of those rows: no row reads another one's result there but through the
// keys and values (6000 rows of an 8B block 2310 us, one of them 260).
//
// Of few rows the q/k/v, output and down products leave their sums in slabs, which the rotation and the next
// norm add up (a block of 8B at 45 rows 122 us, 116 so); of a prompt's first rows the rotation and the attention
// are one launch too: seven a block instead of up to eleven.  Of up to eight narrow rows the gated product norms them
// itself: six.
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
int cake_slab_attn(int dt, const float* ws, int slabs, void* out, long long ldo, int T, int nh, int nkv, int hd,
                   const float* inv_freq, int S, void* kc, void* vc, float scale, hipStream_t st);
int cake_gemm_few_add(int dt, const void* a, long long lda, const void* b, long long ldb, float* r, long long ldr, int M,
                      int N, int K, hipStream_t st);
int cake_gemm_few_gated(int dt, const float* h, long long ldh, const void* ln, float eps, const void* b, long long ldb,
                        void* c, long long ldc, int M, int N, int K, hipStream_t st);
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
  Form kv_form, q1_form, o1_form, gu1_form, down1_form;   // of the last block, with a tail
  int n, dt, T, H, I, nh, nkv, hd, S, pos0;
  int tail;                     // rows of the result that are wanted, the last ones (0: all)
  int few, few1;                // output and gate / up products as cake_gemm_few_*; of the last block, with a tail
  float eps, scale;
};

namespace {

struct Run {
  const CakeBlockRun* r;
  hipStream_t st;
  int nq = r->nh * r->hd, nk = r->nkv * r->hd, nqkv = nq + 2 * nk;
  float* hidden = r->hidden;    // the rows at work: T of them from position pos0 on
  uint16_t* x = static_cast<uint16_t*>(r->x);
  uint16_t* qkv = static_cast<uint16_t*>(r->qkv);
  int T = r->T, pos0 = r->pos0;

  void only_last(int n) {
    const size_t skip = T - n;
    hidden += skip * r->H;
    x += skip * r->H;
    qkv += skip * nqkv;
    pos0 += (int)skip;
    T = n;
  }
  int product(const Form& f, int epi, const void* a, const void* w, void* c, long long ldc, int N, int K) const {
    void* resid = epi == kEpiResid32 ? hidden : nullptr;
    const long long ldr = resid ? N : 0;
    return f.kind ? cake_gemm_rows(r->dt, epi, f.kind, a, K, w, K, c, ldc, nullptr, resid, ldr, r->rows_ws,
                                   r->tick, r->zeros, T, N, K, 1.f, st)
                  : cake_gemm_scaled(r->dt, epi, f.cfg, f.splits, a, K, w, K, c, ldc, nullptr, resid, ldr,
                                     f.splits > 1 ? r->ws : nullptr, r->tick, r->zeros, T, N, K, 1.f, st);
  }
  // the product's slabs, their number (or minus an error)
  int slabs(const Form& f, const void* a, const void* w, int N, int K) const {
    return cake_gemm_slabs(r->dt, f.kind, f.cfg, f.splits, a, K, w, K, r->slabs, r->zeros, T, N, K, st);
  }
  // x = norm of the rows; one norm kernel at every place of a run
  int norm(const void* ln, bool slab) const {
    return slab ? cake_slab_norm(r->dt, nullptr, 0, hidden, r->H, nullptr, 1.f, ln, 0, 0.f, r->eps, 0, T, r->H, x,
                                 r->H, st)
                : cake_rmsnorm(r->dt, hidden, ln, r->eps, T, r->H, x, st);
  }
  // hidden += a w^T, and x = the norm of it by `ln` (null: none)
  int add_norm(const Form& f, const void* a, const void* w, int K, const void* ln) const {
    if (f.slabs) {
      const int n = slabs(f, a, w, r->H, K);
      return n < 0 ? -n : cake_slab_norm(r->dt, r->slabs, n, hidden, r->H, nullptr, 1.f, ln, 0, 0.f, r->eps, 0, T,
                                         r->H, x, r->H, st);
    }
    const int e = product(f, kEpiResid32, a, w, nullptr, 0, r->H, K);
    return e || !ln ? e : cake_rmsnorm(r->dt, hidden, ln, r->eps, T, r->H, x, st);
  }
  // hidden += att wo^T, act = the gated product of its norm: up to eight rows
  int few(const Block& b) const {
    const int e = cake_gemm_few_add(r->dt, r->att, nq, b.wo, nq, hidden, r->H, T, r->H, nq, st);
    return e ? e : cake_gemm_few_gated(r->dt, hidden, r->H, b.ln2, r->eps, b.wgu, r->H, r->act, r->I, T, r->I, r->H, st);
  }
  // rotated heads in qkv (q), keys and values in the cache
  int project(const Block& b) const {
    if (r->qkv_form.slabs) {
      const int n = slabs(r->qkv_form, x, b.wqkv, nqkv, r->H);
      return n < 0 ? -n : cake_slab_rope(r->dt, r->slabs, n, qkv, nqkv, T, r->nh, r->nkv, r->hd, r->inv_freq, pos0,
                                         r->S, b.kc, b.vc, st);
    }
    const int e = product(r->qkv_form, kEpiStore, x, b.wqkv, qkv, nqkv, nqkv, r->H);
    return e ? e : rope(b, r->nh, r->nkv);
  }
  int rope(const Block& b, int nh, int nkv) const {
    return cake_rope_kv(r->dt, qkv, qkv + nq, qkv + nq + nk, nqkv, nqkv, T, nh, nkv, r->hd, r->inv_freq, pos0, r->S,
                        b.kc, b.vc, st);
  }
  // the same, q of the last `tail` rows only, which are the rows at work from here on
  int project_tail(const Block& b) {
    const uint16_t* w = static_cast<const uint16_t*>(b.wqkv);
    int e = product(r->kv_form, kEpiStore, x, w + (size_t)nq * r->H, qkv + nq, nqkv, 2 * nk, r->H);
    if (!e) e = rope(b, 0, r->nkv);
    only_last(r->tail);
    if (!e) e = product(r->q1_form, kEpiStore, x, w, qkv, nqkv, nq, r->H);
    return e ? e : rope(b, r->nh, 0);
  }
  // a short prompt's: projections left in slabs, rotation and attention in one launch
  bool short_prompt() const {
    return r->qkv_form.slabs && pos0 == 0 && T <= 64 && (r->hd == 64 || r->hd == 128);
  }
  int project_attend(const Block& b) const {
    const int n = slabs(r->qkv_form, x, b.wqkv, nqkv, r->H);
    return n < 0 ? -n : cake_slab_attn(r->dt, r->slabs, n, r->att, nq, T, r->nh, r->nkv, r->hd, r->inv_freq, r->S,
                                       b.kc, b.vc, r->scale, st);
  }
  int attend(const Block& b) const {
    const long long Sh = (long long)r->S * r->hd, kv = r->nkv * Sh;
    // [batch, head, row] strides of q (a column block of qkv), the cache twice, the output
    const long long strides[12] = {(long long)T * nqkv, r->hd, nqkv, kv, Sh, r->hd, kv, Sh, r->hd,
                                   (long long)T * nq, r->hd, nq};
    return cake_flash_attn(r->dt, qkv, b.kc, b.vc, r->att, 1, r->nh, r->nkv, T, pos0 + T, r->hd, strides, r->scale,
                           1, pos0, st);
  }
};

}  // namespace

// 0, or the HIP error of the first launch that failed (the blocks behind it are not launched)
CAKE_API int cake_block_rows(const CakeBlockRun* r, hipStream_t st) {
  if (!r || r->n < 0 || r->T < 1 || r->pos0 < 0 || r->pos0 + r->T > r->S || r->tail < 0 || r->tail > r->T)
    return (int)hipErrorInvalidValue;
  Run g{r, st};
  int e = r->n ? g.norm(r->blocks[0].ln1, r->down_form.slabs) : 0;
  for (int i = 0; !e && i < r->n; ++i) {
    const Block& b = r->blocks[i];
    const bool last = i + 1 == r->n, tail = last && r->tail > 0;
    const Form &o = tail ? r->o1_form : r->o_form, &gu = tail ? r->gu1_form : r->gu_form;
    const Form& down = tail ? r->down1_form : r->down_form;
    if (!tail && g.short_prompt()) {
      e = g.project_attend(b);
    } else {
      e = tail ? g.project_tail(b) : g.project(b);
      if (!e) e = g.attend(b);
    }
    if (tail ? r->few1 : r->few) {
      if (!e) e = g.few(b);
    } else {
      if (!e) e = g.add_norm(o, r->att, b.wo, g.nq, b.ln2);
      if (!e) e = g.product(gu, kEpiSwiglu, g.x, b.wgu, r->act, r->I, r->I, r->H);
    }
    if (!e) e = g.add_norm(down, r->act, b.wd, r->I, last ? nullptr : r->blocks[i + 1].ln1);
  }
  return e;
}
