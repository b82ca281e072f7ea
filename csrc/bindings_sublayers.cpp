// Torch op registrations of latent attention, retention, expert mixtures and post-normed sublayers
// (postnorm.hip, latent.hip, latent_mfma.hip, retention.hip, retention_chunk.hip, moe.hip, moe_mfma.hip).  Activations are bf16 or f32; norms, tables,
// recurrent state and the residual stream are f32.
#include "bindings_util.h"
#include "kernels/sublayer.h"

extern "C" {
int mx_post_norm(const mx::PostNorm* a, int f32, hipStream_t stream);
int mx_post_side(const mx::PostNorm* a, const uint16_t* g, const uint16_t* P, int R, hipStream_t stream);
int mx_side_act(const void* z, int64_t ldz, const void* emb, int64_t lde, const int64_t* ids, int V, void* y, int f32,
                int64_t T, int dim, hipStream_t stream);
int mx_side_gate(const uint16_t* x, int64_t ldx, const uint16_t* w, int64_t ldw, const uint16_t* emb, int64_t lde,
                 const int64_t* ids, int V, uint16_t* y, int T, int N, int K, hipStream_t stream);
int mx_post_route(const mx::PostRoute* a, hipStream_t stream);
int mx_clipped_glu(const void* z, int64_t ldz, void* y, int f32, int64_t T, int F, float limit, hipStream_t stream);
int mx_latent_rows(const mx::LatentRows* a, int f32, hipStream_t stream);
int mx_latent_attn(const mx::LatentAttn* a, int f32, hipStream_t stream);
int mx_latent_query(const mx::LatentDecode* a, int f32, hipStream_t stream);
int mx_latent_scan(const mx::LatentDecode* a, int f32, hipStream_t stream);
int mx_latent_value(const mx::LatentDecode* a, int f32, hipStream_t stream);
int mx_retention_seq(const mx::Retention* a, int f32, hipStream_t stream);
int mx_latent_flash(const mx::LatentAttn* a, hipStream_t stream);
int mx_latent_split(const mx::LatentDecode* a, int heads, hipStream_t stream);
int mx_latent_heads(const mx::LatentDecode* a, const mx::LatentRows* rows, int query, hipStream_t stream);
int mx_post_dots(const mx::PostDots* a, hipStream_t stream);
int mx_retention_chunks(const mx::RetentionChunks* a, int f32, hipStream_t stream);
int mx_moe_route_mfma(const uint16_t* x, int64_t ldx, const uint16_t* w, int32_t* ids, float* wts, int T, int K, int E,
                      int top, hipStream_t stream);
int mx_moe_grouped(const mx::MoeGemm* a, int64_t xrows, hipStream_t stream);
int mx_moe_few(const mx::MoeFew* a, int glu, hipStream_t stream);
int mx_moe_route(const void* x, int64_t ldx, const void* w, int f32, int32_t* ids, float* wts, int T, int K, int E,
                 int top, hipStream_t stream);
int mx_moe_group(const int32_t* ids, int P, int top, int E, int bm, int32_t* src, int32_t* inv, int32_t* tiles,
                 int ntiles, hipStream_t stream);
int mx_moe_gemm(const mx::MoeGemm* a, int f32, hipStream_t stream);
}

namespace {

bool is_f32(const at::Tensor& t, const char* name) {
  MX_CHECK(t.is_cuda(), name, " must be a GPU tensor");
  MX_CHECK(t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat, name, " must be bf16 or f32");
  return t.scalar_type() == at::kFloat;
}
// rows [T, n] with unit inner stride, of the activation type: their stride
int64_t rows_of(const at::Tensor& t, const char* name, bool f32, int64_t T, int64_t n) {
  MX_CHECK(is_f32(t, name) == f32, name, " must have the activations' type");
  MX_CHECK(t.dim() == 2 && t.size(0) == T && t.size(1) >= n && (t.stride(1) == 1 || t.size(1) == 1) &&
               (t.stride(0) >= t.size(1) || T == 1),
           name, " must be rows [", T, ", >= ", n, "]");
  return T == 1 ? std::max(t.stride(0), t.size(1)) : t.stride(0);
}
const float* f32_ptr(const at::Tensor& t, const char* name, int64_t n) {
  check_f32(t, name);
  MX_CHECK(t.numel() == n, name, " must have ", n, " elements");
  return t.data_ptr<float>();
}
const int32_t* int_ptr(const at::Tensor& t, const char* name, int64_t n) {
  MX_CHECK(t.is_cuda() && t.scalar_type() == at::kInt && t.is_contiguous() && t.numel() >= n, name,
           " must be a contiguous int32 GPU tensor of at least ", n, " elements");
  return t.data_ptr<int32_t>();
}
const int64_t* id_ptr(const at::Tensor& t, int64_t n) {
  MX_CHECK(t.is_cuda() && t.scalar_type() == at::kLong && t.is_contiguous() && t.numel() == n, "ids int64 [", n, "]");
  return t.data_ptr<int64_t>();
}
// cos / sin [positions, half]
void rope_ptrs(const at::Tensor& cos, const at::Tensor& sin, int64_t half, const float*& c, const float*& s) {
  check_f32(cos, "cos");
  check_f32(sin, "sin");
  MX_CHECK(cos.dim() == 2 && cos.size(1) == half && sin.sizes() == cos.sizes(), "cos / sin [positions, ", half, "]");
  c = cos.data_ptr<float>(), s = sin.data_ptr<float>();
}

// ---- post-normed sublayers
mx::PostNorm pn_args(const at::Tensor& h, const at::Tensor& w, double eps) {
  check_f32(h, "h");
  MX_CHECK(h.dim() == 2, "h [T, W]");
  mx::PostNorm a = {};
  a.T = h.size(0), a.W = (int)h.size(1), a.eps = (float)eps;
  a.h = h.data_ptr<float>();
  a.w = f32_ptr(w, "w", a.W);
  return a;
}
// the bf16 copy of h (f32 activations: empty, h itself serves)
at::Tensor pn_run(mx::PostNorm& a, const at::Tensor& h, bool f) {
  at::Tensor y = f ? at::empty({0}, h.options()) : at::empty_like(h, h.options().dtype(at::kBFloat16));
  a.y = f ? nullptr : y.data_ptr();
  MX_OK(mx_post_norm(&a, f, cur_stream()));
  return y;
}
at::Tensor post_norm(const at::Tensor& src, at::Tensor h, const at::Tensor& w, double eps) {
  DevGuard g(h.device());
  mx::PostNorm a = pn_args(h, w, eps);
  const bool f = is_f32(src, "src");
  a.mode = mx::PostNorm::kRows;
  a.lds = rows_of(src, "src", f, a.T, a.W);
  a.src = src.data_ptr();
  return pn_run(a, h, f);
}
// post_norm of prompt rows and moe_route of its copy (bf16): mx_post_route
std::tuple<at::Tensor, at::Tensor, at::Tensor> post_route(const at::Tensor& src, at::Tensor h, const at::Tensor& w, double eps,
                                                          const at::Tensor& m, int64_t top) {
  DevGuard g(h.device());
  mx::PostRoute a = {};
  a.p = pn_args(h, w, eps);
  a.p.mode = mx::PostNorm::kRows;
  a.p.lds = rows_of(src, "src", false, a.p.T, a.p.W);
  a.p.src = src.data_ptr();
  MX_CHECK(!is_f32(m, "router") && m.dim() == 2 && m.is_contiguous() && m.size(1) == a.p.W && m.device() == h.device() &&
               src.device() == h.device() && w.device() == h.device(), "router [E, W], all on one device");
  MX_CHECK(m.size(0) <= 16 && top >= 1 && top <= m.size(0), "post_route: up to 16 experts");
  a.m = (const uint16_t*)m.data_ptr(), a.E = (int)m.size(0), a.top = (int)top;
  auto y = at::empty({a.p.T, (int64_t)a.p.W}, src.options());
  auto ids = at::empty({a.p.T, top}, src.options().dtype(at::kInt));
  auto wts = at::empty({a.p.T, top}, src.options().dtype(at::kFloat));
  a.p.y = y.data_ptr(), a.ids = ids.data_ptr<int32_t>(), a.wts = wts.data_ptr<float>();
  const int rc = mx_post_route(&a, cur_stream());
  MX_CHECK(rc != -1, "post_route: shape, stride or alignment not taken");
  MX_OK(rc);
  return {y, ids, wts};
}
// bf16 decode rows: h += rms(P g) * w, the copy of h returned; g [T, R], P [W, R]
at::Tensor post_side(const at::Tensor& gs, const at::Tensor& P, at::Tensor h, const at::Tensor& w, double eps) {
  DevGuard g(h.device());
  mx::PostNorm a = pn_args(h, w, eps);
  MX_CHECK(!is_f32(gs, "g") && !is_f32(P, "P") && gs.dim() == 2 && P.dim() == 2 && gs.is_contiguous() && P.is_contiguous() &&
               gs.size(0) == a.T && P.size(0) == a.W && gs.size(1) == P.size(1) && gs.device() == h.device() &&
               P.device() == h.device() && w.device() == h.device(),
           "post_side: g [T, R], P [W, R] bf16, all on one device");
  auto y = at::empty({a.T, (int64_t)a.W}, h.options().dtype(at::kBFloat16));
  a.y = y.data_ptr();
  MX_OK(mx_post_side(&a, (const uint16_t*)gs.data_ptr(), (const uint16_t*)P.data_ptr(), (int)P.size(1), cur_stream()));
  return y;
}
// bf16 decode rows: (new h, its bf16 copy, its dot products with the rows of m) - src a sublayer's rows, or with
// wts [T, top] the experts' rows in pair order (+ the shared expert's).  emb: the products are a gate on columns
// [off, off + rows) of the tokens' rows of emb, and no copy is made
std::tuple<at::Tensor, at::Tensor, at::Tensor> post_dots(const at::Tensor& src, const at::Tensor& h, const at::Tensor& w,
                                                         double eps, const at::Tensor& m, const c10::optional<at::Tensor>& wts,
                                                         const c10::optional<at::Tensor>& shared,
                                                         const c10::optional<at::Tensor>& emb,
                                                         const c10::optional<at::Tensor>& ids, int64_t off) {
  DevGuard g(h.device());
  mx::PostDots a = {};
  a.p = pn_args(h, w, eps);
  mx::PostNorm& p = a.p;
  p.mode = wts.has_value() ? mx::PostNorm::kMix : mx::PostNorm::kRows;
  p.top = 1;
  if (wts.has_value()) {
    check_f32(*wts, "wts");
    MX_CHECK(wts->dim() == 2 && wts->size(0) == p.T && wts->size(1) > 0, "wts [T, top]");
    p.top = (int)wts->size(1), p.wts = wts->data_ptr<float>();
  }
  p.lds = rows_of(src, "src", false, p.T * p.top, p.W);
  p.src = src.data_ptr();
  if (shared.has_value()) p.ldsh = rows_of(*shared, "shared", false, p.T, p.W), p.shared = shared->data_ptr();
  MX_CHECK(!is_f32(m, "m") && m.dim() == 2 && m.is_contiguous() && m.size(1) == p.W, "m [rows, W]");
  a.m = (const uint16_t*)m.data_ptr(), a.R = (int)m.size(0);
  auto ho = at::empty_like(h);
  a.ho = ho.data_ptr<float>();
  at::Tensor y, out;
  if (emb.has_value()) {
    MX_CHECK(ids.has_value() && !is_f32(*emb, "emb") && emb->dim() == 2 && emb->is_contiguous() && off >= 0 &&
                 off + a.R <= emb->size(1),
             "emb [V, >= off + rows]");
    y = at::empty({0}, src.options());
    out = at::empty({p.T, (int64_t)a.R}, src.options());
    a.emb = (const uint16_t*)emb->data_ptr() + off, a.lde = emb->size(1), a.V = (int)emb->size(0), a.ids = id_ptr(*ids, p.T);
    a.side = (uint16_t*)out.data_ptr();
  } else {
    y = at::empty_like(h, src.options());
    out = at::empty({p.T, (int64_t)a.R}, h.options());
    p.y = y.data_ptr();
    a.logits = out.data_ptr<float>();
  }
  MX_OK(mx_post_dots(&a, cur_stream()));
  return {ho, y, out};
}
std::tuple<at::Tensor, at::Tensor> embed_norm(const at::Tensor& ids, const at::Tensor& table, const at::Tensor& w, double eps) {
  DevGuard g(table.device());
  const bool f = is_f32(table, "table");
  MX_CHECK(table.dim() == 2 && table.is_contiguous(), "table [V, W]");
  auto h = at::empty({ids.numel(), table.size(1)}, table.options().dtype(at::kFloat));
  mx::PostNorm a = pn_args(h, w, eps);
  a.mode = mx::PostNorm::kEmbed;
  a.src = table.data_ptr(), a.lds = a.W, a.V = (int)table.size(0), a.ids = id_ptr(ids, a.T);
  auto y = pn_run(a, h, f);
  return {h, y};
}
at::Tensor mix_post_norm(const at::Tensor& src, const c10::optional<at::Tensor>& inv, const at::Tensor& wts,
                         const c10::optional<at::Tensor>& shared, at::Tensor h, const at::Tensor& w, double eps) {
  DevGuard g(h.device());
  mx::PostNorm a = pn_args(h, w, eps);
  const bool f = is_f32(src, "src");
  check_f32(wts, "wts");
  MX_CHECK(wts.dim() == 2 && wts.size(0) == a.T && wts.size(1) > 0, "wts [T, top]");
  a.mode = mx::PostNorm::kMix;
  a.top = (int)wts.size(1), a.wts = wts.data_ptr<float>();
  a.lds = rows_of(src, "src", f, a.T * a.top, a.W);
  a.src = src.data_ptr();
  if (inv.has_value()) a.inv = int_ptr(*inv, "inv", a.T * a.top);
  if (shared.has_value()) a.ldsh = rows_of(*shared, "shared", f, a.T, a.W), a.shared = shared->data_ptr();
  return pn_run(a, h, f);
}
at::Tensor side_act(const at::Tensor& z, const at::Tensor& emb, const at::Tensor& ids, int64_t off) {
  const bool f = is_f32(z, "z");
  DevGuard g(z.device());
  const int64_t T = z.size(0), dim = z.size(1), ldz = rows_of(z, "z", f, T, dim);
  MX_CHECK(is_f32(emb, "emb") == f && emb.dim() == 2 && emb.is_contiguous() && off >= 0 && off + dim <= emb.size(1),
           "emb [V, >= off + dim]");
  auto y = at::empty({T, dim}, z.options());
  MX_OK(mx_side_act(z.data_ptr(), ldz, (const char*)emb.data_ptr() + off * emb.element_size(), emb.size(1), id_ptr(ids, T),
                    (int)emb.size(0), y.data_ptr(), f, T, (int)dim, cur_stream()));
  return y;
}
// side_act(x w^T) of a prompt pass, x [T, K], w [N, K] (bf16): mx_side_gate
at::Tensor side_gate(const at::Tensor& x, const at::Tensor& w, const at::Tensor& emb, const at::Tensor& ids, int64_t off) {
  MX_CHECK(x.is_cuda() && w.device() == x.device() && emb.device() == x.device(), "side_gate: tensors of one GPU");
  MX_CHECK(x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 && emb.scalar_type() == at::kBFloat16,
           "side_gate: bf16 tensors");
  MX_CHECK(x.dim() == 2 && w.dim() == 2 && w.size(1) == x.size(1) && x.stride(1) == 1 && w.stride(1) == 1,
           "side_gate: x [T, K], w [N, K]");
  DevGuard g(x.device());
  const int64_t T = x.size(0), K = x.size(1), N = w.size(0);
  MX_CHECK(emb.dim() == 2 && emb.is_contiguous() && off >= 0 && off + N <= emb.size(1) && emb.size(0) <= INT32_MAX,
           "emb [V, >= off + dim]");
  MX_CHECK(T <= INT32_MAX && N <= INT32_MAX && K <= INT32_MAX, "side_gate: sizes");
  auto y = at::empty({T, N}, x.options());
  const int rc = mx_side_gate((const uint16_t*)x.data_ptr(), x.stride(0), (const uint16_t*)w.data_ptr(), w.stride(0),
                              (const uint16_t*)emb.data_ptr() + off, emb.size(1), id_ptr(ids, T), (int)emb.size(0),
                              (uint16_t*)y.data_ptr(), (int)T, (int)N, (int)K, cur_stream());
  MX_CHECK(rc != -1, "side_gate: shape, stride or alignment not taken");
  MX_OK(rc);
  return y;
}
at::Tensor clipped_glu(const at::Tensor& z, double limit) {
  const bool f = is_f32(z, "z");
  DevGuard g(z.device());
  const int64_t T = z.size(0), F = z.size(1) / 2, ldz = rows_of(z, "z", f, T, 2 * F);
  MX_CHECK(z.size(1) == 2 * F, "z [T, gate | up]");
  auto y = at::empty({T, F}, z.options());
  MX_OK(mx_clipped_glu(z.data_ptr(), ldz, y.data_ptr(), f, T, (int)F, (float)limit, cur_stream()));
  return y;
}

// ---- latent attention
struct Pool {  // cache [blocks or slots, 1, seq, wc]
  const at::Tensor& t;
  const int32_t* bt = nullptr;
  int maxb = 0, seq = 0, wc = 0;
};
Pool pool_of(const at::Tensor& t, const c10::optional<at::Tensor>& bt, bool f32, int64_t ring) {
  MX_CHECK(is_f32(t, "pool") == f32 && t.dim() == 4 && t.size(1) == 1 && t.is_contiguous(), "pool [blocks, 1, rows, width]");
  Pool p{t};
  p.seq = (int)t.size(2), p.wc = (int)t.size(3);
  if (bt.has_value()) {
    MX_CHECK(bt->is_cuda() && bt->scalar_type() == at::kInt && bt->dim() == 2 && bt->is_contiguous(), "block table");
    p.bt = bt->data_ptr<int32_t>(), p.maxb = (int)bt->size(1);
    MX_CHECK(ring > 0 && ring <= INT32_MAX, "ring");
  } else {
    MX_CHECK(ring > 0 && ring <= p.seq, "a slot's rows hold ", p.seq, " positions, not ", ring);
  }
  return p;
}

at::Tensor latent_rows(const at::Tensor& x, const at::Tensor& w, double eps, const at::Tensor& cos, const at::Tensor& sin,
                       int64_t rot, const at::Tensor& rows, int64_t width, const c10::optional<at::Tensor>& pool,
                       const c10::optional<at::Tensor>& bt, int64_t ring) {
  const bool f = is_f32(x, "x");
  DevGuard g(x.device());
  mx::LatentRows a = {};
  a.T = (int)x.size(0), a.rank = (int)w.numel(), a.rot = (int)rot, a.eps = (float)eps;
  a.ldx = rows_of(x, "x", f, a.T, a.rank + rot);
  MX_CHECK(width >= a.rank + rot, "width");
  a.x = x.data_ptr(), a.w = f32_ptr(w, "w", a.rank);
  rope_ptrs(cos, sin, rot / 2, a.cosb, a.sinb);
  a.rows = int_ptr(rows, "rows", 4ll * a.T);
  auto lat = at::empty({a.T, width}, x.options());
  a.lat = lat.data_ptr(), a.ldl = width;
  if (pool.has_value()) {
    const Pool p = pool_of(*pool, bt, f, ring);
    MX_CHECK(p.wc >= a.rank + rot, "pool rows too narrow");
    a.pool = pool->data_ptr(), a.bt = p.bt, a.maxb = p.maxb, a.seq = p.seq, a.wc = p.wc, a.ring = (int)ring;
  }
  MX_OK(mx_latent_rows(&a, f, cur_stream()));
  return lat;
}

mx::LatentAttn la_args(const at::Tensor& q, const at::Tensor& kv, const at::Tensor& lat, const at::Tensor& cos,
                       const at::Tensor& sin, const c10::optional<at::Tensor>& sink, int64_t H, int64_t D, int64_t R,
                       int64_t E, int64_t rank, int64_t window, double scale) {
  const bool f = is_f32(q, "q");
  const int64_t T = q.size(0);
  MX_CHECK(H > 0 && D > 0 && R >= 0 && R % 2 == 0 && E > 0 && rank > 0 && window >= 0 && window <= INT32_MAX, "latent attention sizes");
  mx::LatentAttn a = {};
  a.ldq = rows_of(q, "q", f, T, H * (D + R)), a.ldkv = rows_of(kv, "kv", f, T, H * (D + E));
  a.ldl = rows_of(lat, "lat", f, T, rank + R);
  a.q = q.data_ptr(), a.kv = kv.data_ptr(), a.lat = lat.data_ptr();
  rope_ptrs(cos, sin, R / 2, a.cosb, a.sinb);
  if (sink.has_value()) a.sink = f32_ptr(*sink, "sink", H);
  a.T = (int)T, a.H = (int)H, a.D = (int)D, a.R = (int)R, a.E = (int)E, a.rank = (int)rank, a.window = (int)window;
  a.scale = (float)scale;
  return a;
}
at::Tensor latent_attn(const at::Tensor& q, const at::Tensor& kv, const at::Tensor& lat, const at::Tensor& cos,
                       const at::Tensor& sin, const at::Tensor& rows, const c10::optional<at::Tensor>& blocks,
                       const c10::optional<at::Tensor>& sink, int64_t H, int64_t D, int64_t R, int64_t E, int64_t rank,
                       int64_t window, double scale) {
  DevGuard g(q.device());
  mx::LatentAttn a = la_args(q, kv, lat, cos, sin, sink, H, D, R, E, rank, window, scale);
  a.rows = int_ptr(rows, "rows", 4ll * a.T);
  auto o = at::empty({(int64_t)a.T, H * E}, q.options());
  a.out = o.data_ptr();
  const bool f = is_f32(q, "q");
  if (!f && blocks.has_value()) {  // matrix cores, where they take the sizes
    a.nblocks = (int)blocks->size(0);
    a.blocks = int_ptr(*blocks, "blocks", 4ll * a.nblocks);
    const int rc = mx_latent_flash(&a, cur_stream());
    if (rc != -1) {
      MX_OK(rc);
      return o;
    }
  }
  MX_OK(mx_latent_attn(&a, f, cur_stream()));
  return o;
}

// one query per sequence against the cache: q [B, H (D + R)], wkv [H D + H E, rank]; max_len bounds the visible
// keys.  own_x [B, rank + R], own_w: the new tokens' latents, stored first.  wuk_t [H, rank, D]: W_uk transposed
// (bf16: the products per head on the matrix cores)
at::Tensor latent_decode(const at::Tensor& q, const at::Tensor& wkv, const at::Tensor& cos, const at::Tensor& sin,
                         const at::Tensor& pos, const at::Tensor& slots, const at::Tensor& pool,
                         const c10::optional<at::Tensor>& bt, int64_t ring, const c10::optional<at::Tensor>& sink,
                         int64_t H, int64_t D, int64_t R, int64_t E, int64_t rank, int64_t window, double scale,
                         int64_t max_len, const c10::optional<at::Tensor>& own_x, const c10::optional<at::Tensor>& own_w,
                         double eps, const c10::optional<at::Tensor>& wuk_t) {
  const bool f = is_f32(q, "q");
  DevGuard g(q.device());
  const int64_t B = q.size(0);
  MX_CHECK(H > 0 && D > 0 && R >= 0 && R % 2 == 0 && E > 0 && rank > 0 && window >= 0 && window <= INT32_MAX && max_len > 0,
           "latent attention sizes");
  MX_CHECK(is_f32(wkv, "wkv") == f && wkv.is_contiguous() && wkv.dim() == 2 && wkv.size(0) == H * (D + E) && wkv.size(1) == rank,
           "wkv [H (D + E), rank]");
  const Pool p = pool_of(pool, bt, f, ring);
  mx::LatentDecode a = {};
  a.ldq = rows_of(q, "q", f, B, H * (D + R));
  a.q = q.data_ptr(), a.wuk = wkv.data_ptr(), a.wuv = (const char*)wkv.data_ptr() + H * D * rank * wkv.element_size();
  rope_ptrs(cos, sin, R / 2, a.cosb, a.sinb);
  a.pos = int_ptr(pos, "pos", B), a.slots = int_ptr(slots, "slots", B);
  a.pool = pool.data_ptr(), a.bt = p.bt, a.maxb = p.maxb, a.seq = p.seq, a.wc = p.wc, a.ring = (int)ring;
  if (sink.has_value()) a.sink = f32_ptr(*sink, "sink", H);
  a.B = (int)B, a.H = (int)H, a.D = (int)D, a.R = (int)R, a.E = (int)E, a.rank = (int)rank, a.window = (int)window;
  a.scale = (float)scale;
  a.wq = p.wc;
  const int64_t keys = window > 0 ? std::min(window, max_len) : max_len;
  // matrix cores: 32 heads a workgroup, 16 where that leaves the GPU empty, and keys split in runs of 64 to 512
  // so that there are about two workgroups for every CU
  const bool mfma = !f && rank % 4 == 0 && a.wc % 32 == 0 && a.wc <= 1024 && scale > 0;
  int heads = H <= 16 || a.wc > 768 || B * ((keys + 63) / 64) * ((H + 31) / 32) < 256 ? 16 : 32;
  const int64_t per = B * ((H + heads - 1) / heads), want = std::max<int64_t>(1, 512 / per);
  a.span = mfma ? (int)std::min<int64_t>(512, std::max<int64_t>(64, ((keys + want - 1) / want + 31) / 32 * 32)) : 256;
  a.nsplit = (int)((keys + a.span - 1) / a.span);
  auto qa = at::empty({B, H, (int64_t)a.wq}, q.options());
  auto ml = at::empty({B, H, (int64_t)a.nsplit, 2}, q.options().dtype(at::kFloat));
  auto po = at::empty({B, H, (int64_t)a.nsplit, rank}, q.options().dtype(at::kFloat));
  auto out = at::empty({B, H * E}, q.options());
  a.qa = qa.data_ptr(), a.ml = ml.data_ptr<float>(), a.po = po.data_ptr<float>(), a.out = out.data_ptr();
  mx::LatentRows rw = {};
  if (own_x.has_value()) {
    MX_CHECK(own_w.has_value(), "own_w");
    rw.T = (int)B, rw.rank = (int)rank, rw.rot = (int)R, rw.eps = (float)eps;
    rw.ldx = rows_of(*own_x, "own_x", f, B, rank + R);
    rw.x = own_x->data_ptr(), rw.w = f32_ptr(*own_w, "own_w", rank);
    rw.cosb = a.cosb, rw.sinb = a.sinb;
    rw.pool = pool.data_ptr(), rw.bt = p.bt, rw.maxb = p.maxb, rw.seq = p.seq, rw.wc = p.wc, rw.ring = (int)ring;
    MX_CHECK(p.wc >= rank + R, "pool rows too narrow");
  }
  int rc = -1;
  at::Tensor om;
  if (wuk_t.has_value() && mfma) {
    MX_CHECK(!is_f32(*wuk_t, "wuk_t") && wuk_t->is_contiguous() && wuk_t->numel() == H * D * rank, "wuk_t [H, rank, D]");
    om = at::empty({B, H, rank}, q.options());
    a.wuk_t = wuk_t->data_ptr(), a.om = om.data_ptr();
    if (a.nsplit <= 1024) rc = mx_latent_heads(&a, &rw, 1, cur_stream());
    if (rc != -1) {
      MX_OK(rc);
      MX_OK(mx_latent_split(&a, heads, cur_stream()));
      MX_OK(mx_latent_heads(&a, nullptr, 0, cur_stream()));
      return out;
    }
  }
  at::Tensor info;
  if (rw.x) {
    info = at::stack({pos, slots, pos + 1, pos}, 1).contiguous();
    rw.rows = info.data_ptr<int32_t>();
    MX_OK(mx_latent_rows(&rw, f, cur_stream()));
  }
  MX_OK(mx_latent_query(&a, f, cur_stream()));
  if (mfma) MX_OK(mx_latent_split(&a, heads, cur_stream()));
  else MX_OK(mx_latent_scan(&a, f, cur_stream()));
  MX_OK(mx_latent_value(&a, f, cur_stream()));
  return out;
}

// ---- retention: x [T, q | k | v | gate]; prompts by seqs [n, 4], else one token a row
at::Tensor retention(const at::Tensor& x, const at::Tensor& decay, const at::Tensor& cos, const at::Tensor& sin, int64_t rd,
                     int64_t D, int64_t E, double eps, const c10::optional<at::Tensor>& seqs,
                     const c10::optional<at::Tensor>& pos, const c10::optional<at::Tensor>& slots,
                     c10::optional<at::Tensor> state) {
  const bool f = is_f32(x, "x");
  DevGuard g(x.device());
  check_f32(decay, "decay");
  MX_CHECK(decay.dim() == 2 && decay.size(1) >= 2, "decay [H, powers]");
  const int64_t H = decay.size(0), T = x.size(0);
  mx::Retention a = {};
  a.ldx = rows_of(x, "x", f, T, 2 * H * (D + E));
  a.x = x.data_ptr(), a.decay = decay.data_ptr<float>() + 1, a.ldd = decay.size(1), a.eps = (float)eps;
  rope_ptrs(cos, sin, rd / 2, a.cosb, a.sinb);
  a.T = (int)T, a.H = (int)H, a.D = (int)D, a.E = (int)E, a.rd = (int)rd;
  if (seqs.has_value()) {
    a.nseq = (int)seqs->size(0);
    a.seqs = int_ptr(*seqs, "seqs", 4ll * a.nseq);
  } else {
    MX_CHECK(pos.has_value() && slots.has_value() && state.has_value(), "a token needs its position, slot and state");
    a.pos = int_ptr(*pos, "pos", T), a.slots = int_ptr(*slots, "slots", T);
  }
  if (state.has_value()) {
    check_f32(*state, "state");
    MX_CHECK(state->dim() == 2 && state->size(1) == H * D * E, "state [slots, H D E]");
    a.state = state->data_ptr<float>();
  }
  auto y = at::empty({T, H * E}, x.options());
  a.y = y.data_ptr();
  MX_OK(mx_retention_seq(&a, f, cur_stream()));
  return y;
}

// prompts in runs of rows (chunks, seqs, blocks: sublayer.h RetentionChunks); D, E <= 256
at::Tensor retention_chunks(const at::Tensor& x, const at::Tensor& powers, const at::Tensor& cos, const at::Tensor& sin,
                            int64_t rd, int64_t D, int64_t E, double eps, const at::Tensor& chunks, const at::Tensor& seqs,
                            const at::Tensor& blocks, bool multi, c10::optional<at::Tensor> state) {
  const bool f = is_f32(x, "x");
  DevGuard g(x.device());
  const int64_t H = powers.size(0), T = x.size(0);
  mx::RetentionChunks a = {};
  a.ldx = rows_of(x, "x", f, T, 2 * H * (D + E));
  a.x = x.data_ptr(), a.pw = f32_ptr(powers, "powers", H * 257), a.eps = (float)eps;
  rope_ptrs(cos, sin, rd / 2, a.cosb, a.sinb);
  a.H = (int)H, a.D = (int)D, a.E = (int)E, a.rd = (int)rd;
  a.nchunks = (int)chunks.size(0), a.nseq = (int)seqs.size(0), a.nblocks = (int)blocks.size(0);
  a.chunks = int_ptr(chunks, "chunks", 4ll * a.nchunks), a.seqs = int_ptr(seqs, "seqs", 4ll * a.nseq);
  a.blocks = int_ptr(blocks, "blocks", 4ll * a.nblocks);
  a.carry = multi || state.has_value();
  auto ws = at::empty({a.carry ? a.nchunks * H * D * E : 0}, x.options().dtype(at::kFloat));
  a.ws = ws.data_ptr<float>();
  if (state.has_value()) {
    check_f32(*state, "state");
    MX_CHECK(state->dim() == 2 && state->size(1) == H * D * E, "state [slots, H D E]");
    a.state = state->data_ptr<float>();
  }
  auto y = at::empty({T, H * E}, x.options());
  a.y = y.data_ptr();
  MX_OK(mx_retention_chunks(&a, f, cur_stream()));
  return y;
}

// ---- mixture of experts
std::tuple<at::Tensor, at::Tensor> moe_route(const at::Tensor& x, const at::Tensor& w, int64_t top) {
  const bool f = is_f32(x, "x");
  DevGuard g(x.device());
  const int64_t T = x.size(0), K = w.size(1), E = w.size(0), ldx = rows_of(x, "x", f, T, K);
  MX_CHECK(is_f32(w, "w") == f && w.dim() == 2 && w.is_contiguous() && x.size(1) == K, "router [E, K]");
  auto ids = at::empty({T, top}, x.options().dtype(at::kInt));
  auto wts = at::empty({T, top}, x.options().dtype(at::kFloat));
  if (!f && T > 16) {  // matrix cores, where they take the sizes
    const int rc = mx_moe_route_mfma((const uint16_t*)x.data_ptr(), ldx, (const uint16_t*)w.data_ptr(), ids.data_ptr<int32_t>(),
                                     wts.data_ptr<float>(), (int)T, (int)K, (int)E, (int)top, cur_stream());
    if (rc != -1) {
      MX_OK(rc);
      return {ids, wts};
    }
  }
  MX_OK(mx_moe_route(x.data_ptr(), ldx, w.data_ptr(), f, ids.data_ptr<int32_t>(), wts.data_ptr<float>(), (int)T, (int)K,
                     (int)E, (int)top, cur_stream()));
  return {ids, wts};
}
// ids [T, top] -> src [T top] (token of each sorted row), inv [T top] (sorted row of each pair), tiles [n, 4] of bm rows
std::tuple<at::Tensor, at::Tensor, at::Tensor> moe_group(const at::Tensor& ids, int64_t E, int64_t bm) {
  const int64_t P = ids.numel(), top = ids.size(1), nt = P / bm + std::min(E, P);
  DevGuard g(ids.device());
  MX_CHECK(P < INT32_MAX / 2, "too many rows for one pass");
  auto src = at::empty({P}, ids.options()), inv = at::empty({P}, ids.options()), tiles = at::empty({nt, 4}, ids.options());
  MX_OK(mx_moe_group(int_ptr(ids, "ids", P), (int)P, (int)top, (int)E, (int)bm, src.data_ptr<int32_t>(), inv.data_ptr<int32_t>(),
                     tiles.data_ptr<int32_t>(), (int)nt, cur_stream()));
  return {src, inv, tiles};
}
mx::MoeGemm mg_args(const at::Tensor& x, const c10::optional<at::Tensor>& src, const at::Tensor& tiles, const at::Tensor& w,
                    int64_t P, bool glu, double limit) {
  const bool f = is_f32(x, "x");
  MX_CHECK(is_f32(w, "w") == f && w.dim() == 3 && w.is_contiguous() && (!glu || w.size(1) % 2 == 0), "w [experts, N, K]");
  mx::MoeGemm a = {};
  a.K = (int)w.size(2), a.N = (int)(glu ? w.size(1) / 2 : w.size(1)), a.glu = glu, a.limit = (float)limit;
  a.ldx = rows_of(x, "x", f, x.size(0), a.K);
  a.x = x.data_ptr(), a.w = w.data_ptr();
  if (src.has_value()) a.src = int_ptr(*src, "src", P);
  else MX_CHECK(x.size(0) == P, "one row of x for every sorted row");
  a.ntiles = (int)tiles.size(0);
  a.tiles = int_ptr(tiles, "tiles", 4ll * a.ntiles);
  return a;
}
// rows sorted by expert through their experts' weights, tiles of bm rows (256: matrix cores, else 64);
// glu: w = [experts, gate | up, K]
at::Tensor moe_gemm(const at::Tensor& x, const c10::optional<at::Tensor>& src, const at::Tensor& tiles, const at::Tensor& w,
                    int64_t P, bool glu, double limit, int64_t bm) {
  MX_CHECK(bm == 64 || bm == 256, "tiles of 64 or 256 rows");
  DevGuard g(x.device());
  mx::MoeGemm a = mg_args(x, src, tiles, w, P, glu, limit);
  auto y = at::empty({P, (int64_t)a.N}, x.options());
  a.y = y.data_ptr();
  if (bm == 256) {
    MX_CHECK(!is_f32(x, "x"), "the matrix-core products are bf16");
    MX_OK(mx_moe_grouped(&a, x.size(0), cur_stream()));
  } else {
    MX_OK(mx_moe_gemm(&a, is_f32(x, "x"), cur_stream()));
  }
  return y;
}
// up to 64 tokens, bf16: x [T, K] (glu) or [T top, K] through each pair's expert -> [T top, N]; the shared
// expert's weights sw on x (glu) or sx -> [T, N'].  Choices: ids, or (glu) the top of f32 logits [T, experts].
// Returns (y, shared y, ids, the choices' weights where logits are given)
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> moe_few(
    const at::Tensor& x, const c10::optional<at::Tensor>& given, const c10::optional<at::Tensor>& logits, int64_t top,
    const at::Tensor& w, bool glu, double limit, const c10::optional<at::Tensor>& sw, const c10::optional<at::Tensor>& sx,
    double slimit) {
  DevGuard g(x.device());
  MX_CHECK(given.has_value() != logits.has_value(), "ids or logits");
  const int64_t T = given.has_value() ? given->size(0) : logits->size(0), G = glu ? 2 : 1;
  at::Tensor ids = given.has_value() ? *given : at::empty({T, top}, x.options().dtype(at::kInt)), wts;
  MX_CHECK(ids.dim() == 2 && ids.size(1) == top, "ids [T, top]");
  MX_CHECK(!is_f32(x, "x") && !is_f32(w, "w") && w.dim() == 3 && w.is_contiguous() && w.size(1) % G == 0, "w [experts, N, K] bf16");
  mx::MoeFew a = {};
  a.T = (int)T, a.top = (int)top, a.E = (int)w.size(0), a.N = (int)(w.size(1) / G), a.K = (int)w.size(2);
  a.limit = (float)limit, a.slimit = (float)slimit;
  a.ldx = rows_of(x, "x", false, glu ? T : T * top, a.K);
  a.x = (const uint16_t*)x.data_ptr(), a.w = (const uint16_t*)w.data_ptr(), a.ids = int_ptr(ids, "ids", T * top);
  if (logits.has_value()) {
    a.logits = f32_ptr(*logits, "logits", T * a.E);
    wts = at::empty({T, top}, logits->options());
    a.ids_out = ids.data_ptr<int32_t>(), a.wts_out = wts.data_ptr<float>();
  } else {
    wts = at::empty({0}, x.options().dtype(at::kFloat));
  }
  auto y = at::empty({T * top, (int64_t)a.N}, x.options());
  a.y = (uint16_t*)y.data_ptr();
  at::Tensor sy = at::empty({0, 0}, x.options());
  if (sw.has_value()) {
    MX_CHECK(!is_f32(*sw, "sw") && sw->dim() == 2 && sw->is_contiguous() && sw->size(0) % G == 0, "sw [N, K] bf16");
    a.sN = (int)(sw->size(0) / G), a.sK = (int)sw->size(1), a.sw = (const uint16_t*)sw->data_ptr();
    if (glu) {
      MX_CHECK(a.sK == a.K, "the shared expert reads the same rows");
    } else {
      MX_CHECK(sx.has_value() && !is_f32(*sx, "sx") && sx->is_contiguous() && sx->dim() == 2 && sx->size(0) == T && sx->size(1) == a.sK,
               "sx [T, K']");
      a.sx = (const uint16_t*)sx->data_ptr();
    }
    sy = at::empty({T, (int64_t)a.sN}, x.options());
    a.sy = (uint16_t*)sy.data_ptr();
  }
  MX_OK(mx_moe_few(&a, glu, cur_stream()));
  return {y, sy, ids, wts};
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(mxllm, m) {
  m.def("post_norm(Tensor src, Tensor(a!) h, Tensor w, float eps) -> Tensor");
  m.def("embed_norm(Tensor ids, Tensor table, Tensor w, float eps) -> (Tensor, Tensor)");
  m.def("post_side(Tensor g, Tensor P, Tensor(a!) h, Tensor w, float eps) -> Tensor");
  m.def("mix_post_norm(Tensor src, Tensor? inv, Tensor wts, Tensor? shared, Tensor(a!) h, Tensor w, float eps) -> Tensor");
  m.def("post_route(Tensor src, Tensor(a!) h, Tensor w, float eps, Tensor m, int top) -> (Tensor, Tensor, Tensor)");
  m.def("side_act(Tensor z, Tensor emb, Tensor ids, int off) -> Tensor");
  m.def("side_gate(Tensor x, Tensor w, Tensor emb, Tensor ids, int off) -> Tensor");
  m.def("clipped_glu(Tensor z, float limit) -> Tensor");
  m.def("latent_rows(Tensor x, Tensor w, float eps, Tensor cos, Tensor sin, int rot, Tensor rows, int width, Tensor(a!)? pool=None, Tensor? bt=None, int ring=0) -> Tensor");
  m.def("latent_attn(Tensor q, Tensor kv, Tensor lat, Tensor cos, Tensor sin, Tensor rows, Tensor? blocks, Tensor? sink, int H, int D, int R, int E, int rank, int window, float scale) -> Tensor");
  m.def("latent_decode(Tensor q, Tensor wkv, Tensor cos, Tensor sin, Tensor pos, Tensor slots, Tensor(a!) pool, Tensor? bt, int ring, Tensor? sink, int H, int D, int R, int E, int rank, int window, float scale, int max_len, Tensor? own_x=None, Tensor? own_w=None, float eps=0., Tensor? wuk_t=None) -> Tensor");
  m.def("post_dots(Tensor src, Tensor h, Tensor w, float eps, Tensor m, Tensor? wts=None, Tensor? shared=None, Tensor? emb=None, Tensor? ids=None, int off=0) -> (Tensor, Tensor, Tensor)");
  m.def("retention(Tensor x, Tensor decay, Tensor cos, Tensor sin, int rd, int D, int E, float eps, Tensor? seqs=None, Tensor? pos=None, Tensor? slots=None, Tensor(a!)? state=None) -> Tensor");
  m.def("moe_route(Tensor x, Tensor w, int top) -> (Tensor, Tensor)");
  m.def("moe_group(Tensor ids, int E, int bm) -> (Tensor, Tensor, Tensor)");
  m.def("moe_gemm(Tensor x, Tensor? src, Tensor tiles, Tensor w, int P, bool glu, float limit, int bm) -> Tensor");
  m.def("moe_few(Tensor x, Tensor? ids, Tensor? logits, int top, Tensor w, bool glu, float limit, Tensor? sw, Tensor? sx, float slimit) -> (Tensor, Tensor, Tensor, Tensor)");
  m.def("retention_chunks(Tensor x, Tensor powers, Tensor cos, Tensor sin, int rd, int D, int E, float eps, Tensor chunks, Tensor seqs, Tensor blocks, bool multi, Tensor(a!)? state=None) -> Tensor");
}

TORCH_LIBRARY_IMPL(mxllm, CUDA, m) {
  m.impl("post_norm", &post_norm);
  m.impl("embed_norm", &embed_norm);
  m.impl("post_side", &post_side);
  m.impl("mix_post_norm", &mix_post_norm);
  m.impl("post_route", &post_route);
  m.impl("side_act", &side_act);
  m.impl("side_gate", &side_gate);
  m.impl("clipped_glu", &clipped_glu);
  m.impl("latent_rows", &latent_rows);
  m.impl("latent_attn", &latent_attn);
  m.impl("latent_decode", &latent_decode);
  m.impl("retention", &retention);
  m.impl("moe_route", &moe_route);
  m.impl("moe_group", &moe_group);
  m.impl("moe_gemm", &moe_gemm);
  m.impl("moe_few", &moe_few);
  m.impl("retention_chunks", &retention_chunks);
  m.impl("post_dots", &post_dots);
}
