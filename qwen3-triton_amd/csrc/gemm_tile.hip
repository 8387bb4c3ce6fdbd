// q3_gemm: the tile and split plan of gemm_tile.h, its K-split combining passes and its C entry points.
#include <algorithm>

#include "gemm_tile.h"

namespace q3gemm {
int launch_tile_nt(int dtype, int cfg, int epi, const Args& a, hipStream_t s);
int launch_tile_nn(int dtype, int cfg, int epi, const Args& a, hipStream_t s);
int launch_tile_tn(int dtype, int cfg, const Args& a, hipStream_t s);
}  // namespace q3gemm

namespace {

using q3gemm::Args;

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }
int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---------------------------------------------------------------- plan
// Tile configurations: rows, columns, workgroups resident per CU (LDS), and the measured time of one 64-wide
// k-tile of one workgroup (us) -- alone on its CU, and with every slot of the chip taken.
struct Cfg {
  int bm, bn, conc;
  double solo, full;
};
constexpr int kNumCfg = 8;
constexpr Cfg kCfg[kNumCfg] = {{256, 256, 1, 1.27, 1.48}, {128, 256, 1, 0.86, 0.94}, {128, 128, 1, 0.48, 0.62},
                               {64, 128, 1, 0.28, 0.32},  {64, 64, 2, 0.34, 0.70},   {32, 64, 3, 0.27, 1.04},
                               {192, 256, 1, 0.98, 1.25}, {192, 128, 1, 0.61, 0.68}};
// Instantiated layouts: the 192-row tiles for a k-contiguous A (they fill the CUs where 256 rows would leave the
// last row of tiles half empty: 1500 x 24576 x 4096 247 against 279 us), 32 rows for two k-contiguous operands.
bool cfg_for(int c, bool at, bool bt) { return c < 5 || (c == 5 ? !bt : !at); }
constexpr int kSplits[6] = {1, 2, 3, 4, 6, 8};
constexpr int64_t kMinSplitK = 512;  // k per split

struct Plan {
  int cfg, splits;
};

// Estimated time of a configuration (us): whole rounds of resident workgroups at the full rate, a last round
// that takes at least a lone workgroup's time, no less than the B operand streamed once at 6 TB/s, and for a K
// split the partial products written and combined.  The constants are a fit to timings on MI355X; measured again
// over 225 shapes (k contiguous / K-major operands, M 17-4096, N 1024-24576, K 64-12288; 4063 timings) the plan it
// picks is 1.7 % slower on average than the best of all configurations and splits, 7 % at the 90th percentile, 26 %
// at worst (512 x 1024 x 1024: 8.3 against 6.6 us).  The order matters more than the values: 256 x 256 tiles sustain
// 1.38-1.45 PFLOP/s once they fill the CUs, smaller tiles and splits keep the CUs busy below that (65 x 4096 x 4096:
// 15 us against 47 us on 32 tiles of 128 x 128).
double estimate(int c, int splits, int64_t tiles, int64_t M, int64_t N, int64_t K, double combine) {
  const Cfg& f = kCfg[c];
  const int64_t w = tiles * splits, slots = 256 * f.conc;
  const int64_t kt = cdiv(cdiv(K, 64), splits), r = w / slots, rem = w % slots;
  const double last = rem ? std::max(f.solo, f.full * (double)rem / (double)slots) : 0.0;
  double t = 5.6 + (double)kt * ((double)r * f.full + last);
  t = std::max(t, 5.6 + 2.0 * (double)N * (double)K / 6e6);
  return splits > 1 ? t + combine + (double)splits * (double)M * (double)N * 4.0 / 5e6 : t;
}

// Tiles of a call along its rows / columns: every piece starts a tile of its own.
int64_t tile_rows(const Args& a, int bm) {
  if (a.axis != 3) return cdiv(a.M, bm);
  int64_t t = 0;
  for (int i = 0; i < a.pieces; ++i) t += cdiv(a.len[i], bm);
  return t;
}
int64_t tile_cols(const Args& a, int bn) {
  if (a.axis != 2) return cdiv(a.N, bn);
  int64_t t = 0;
  for (int i = 0; i < a.pieces; ++i) t += cdiv(a.len[i], bn);
  return t;
}

// combine: what the combining pass adds besides its traffic (us): a launch (4.5 measured on small products), or
// next to nothing where the pass also forms the norm that an unsplit product would leave to a launch of its own.
// can_split: the product may be formed as partial products (plain or residual epilogue, 16-byte columns).
Plan plan_for(const Args& a, bool at, bool bt, bool can_split, double combine) {
  Plan best{0, 1};
  double best_t = 0.0;
  for (int c = 0; c < kNumCfg; ++c) {
    if (!cfg_for(c, at, bt)) continue;
    if (kCfg[c].bm >= 2 * a.M && kCfg[c].bm > (bt ? 64 : 32)) continue;  // more than half of the tile's rows empty
    const int64_t tiles = tile_rows(a, kCfg[c].bm) * tile_cols(a, kCfg[c].bn);
    for (int sp : kSplits) {
      // a grid that fills the chip by itself is not split: its partial products would outgrow the caches
      // (6144 x 4096 x 8192 in two splits: 390 + 43 us against 300 us in two launches, below)
      if (sp > 1 && (!can_split || a.K / sp < kMinSplitK || tiles >= 256 * kCfg[c].conc)) break;
      const double t = estimate(c, sp, tiles, a.M, a.N, a.K, combine);
      if (best_t == 0.0 || t < best_t) {
        best = {c, sp};
        best_t = t;
      }
    }
  }
  return best;
}

// ---------------------------------------------------------------- combining passes
// Sum of the fp32 partial products of one 8-column chunk, rounded to T.
template <typename T> Q3_DEV Vec<T> sum_parts(const float* p, int splits, int64_t ld) {
  f32x4 s0 = *reinterpret_cast<const f32x4*>(p), s1 = *reinterpret_cast<const f32x4*>(p + 4);
  for (int i = 1; i < splits; ++i) {
    p += ld;
    s0 += *reinterpret_cast<const f32x4*>(p);
    s1 += *reinterpret_cast<const f32x4*>(p + 4);
  }
  Vec<T> r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r.v[e] = to_f32<T>(from_f32<T>(e < 4 ? s0[e] : s1[e - 4]));
  return r;
}
template <typename T> Q3_DEV void add_res(Vec<T>& v, const u16* res) {
  const Vec<T> b = load_vec<T>(res);
#pragma unroll
  for (int e = 0; e < 8; ++e) v.v[e] = to_f32<T>(from_f32<T>(v.v[e] + b.v[e]));
}

// C = (res +) the sum of the partial products, with the unsplit epilogue's roundings (the product rounded to
// T, the residual added in fp32, rounded again).  Bound by the partials' traffic, which the GEMM has just
// written (L2 / MALL resident): one 8-column chunk per thread.
template <typename T> __global__ __launch_bounds__(256) void combine_kernel(Args a) {
  const int64_t cols = a.N / 8, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.M * cols) return;
  int64_t r = i / cols, c = (i - r * cols) * 8;
  Vec<T> v = sum_parts<T>(a.part + r * a.N + c, a.splits, a.M * a.N);
  int s = 0;
  int64_t beg = 0;
  if (a.axis >= 2) {
    const int64_t at = a.axis == 2 ? c : r;
    while (s + 1 < a.pieces && at >= beg + a.len[s]) beg += a.len[s++];
    (a.axis == 2 ? c : r) -= beg;
  }
  if (a.res) add_res<T>(v, a.res + r * a.ldres + c);
  store_vec<T>(reinterpret_cast<u16*>(a.c[s]) + r * a.ldc[s] + c, v);
}

// The same for one whole row per 512-thread workgroup (N <= 8192), also writing
// Y = C rsqrt(mean(C^2) + eps) w, the RMSNorm that follows (from the rounded C, one rounding).
template <typename T>
__global__ __launch_bounds__(512) void combine_norm_kernel(Args a, const u16* __restrict__ w, float eps,
                                                           u16* __restrict__ Y, int64_t ldy) {
  constexpr int G = 2;
  __shared__ float red[8];
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x, N = (int)a.N;
  Vec<T> c[G];
  float ss = 0.f;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int col = (g * 512 + tid) * 8;
    if (col >= N) continue;
    c[g] = sum_parts<T>(a.part + r * N + col, a.splits, a.M * a.N);
    if (a.res) add_res<T>(c[g], a.res + r * a.ldres + col);
    store_vec<T>(reinterpret_cast<u16*>(a.c[0]) + r * a.ldc[0] + col, c[g]);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += c[g].v[e] * c[g].v[e];
  }
  ss = group_sum<64>(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) tot += red[i];
  const float inv = rsqrtf(tot * (1.f / (float)N) + eps);
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int col = (g * 512 + tid) * 8;
    if (col >= N) continue;
    const Vec<T> wv = load_vec<T>(w + col);
    Vec<T> o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o.v[e] = c[g].v[e] * inv * wv.v[e];
    store_vec<T>(Y + r * ldy + col, o);
  }
}

// ---------------------------------------------------------------- descriptor -> arguments
struct Call {
  Args a;
  double combine;
  bool at, bt, can_split;
  int epi;
};

bool operand_ok(const void* p, int64_t ld, int64_t rows, int64_t k, bool kmajor) {
  // 16-byte chunks: the contiguous extent (k, or the operand's own index when K-major) and the row stride are
  // whole chunks; a tile's offsets fit the 2^31-byte range of a buffer descriptor
  const int64_t ext = kmajor ? rows : k;
  return p && al16(p) && ld % 8 == 0 && ext % 8 == 0 && ld >= ext && ld < (1 << 22);
}

bool parse(const q3_gemm_desc* d, Call& c) {
  if (!d || (d->dtype != Q3_BF16 && d->dtype != Q3_F16)) return false;
  if (d->m < 1 || d->n < 1 || d->k < 1 || d->m >= (1ll << 31) - 256 || d->n >= (1ll << 30) || d->k >= (1ll << 31) - 256)
    return false;
  if (d->axis < 0 || d->axis > 3 || (d->axis == 0 ? d->pieces != 1 : (d->pieces < 1 || d->pieces > 3))) return false;
  Args& a = c.a;
  a = Args{};
  c.at = d->a_kmajor != 0;
  c.bt = d->b_kmajor != 0;
  if (c.at && !c.bt) return false;
  a.axis = d->axis;
  a.pieces = d->pieces;
  a.M = d->m;
  a.K = d->k;
  a.splits = 1;
  const bool gate_up = d->epilogue == Q3_GEMM_GATE_UP, sbwd = d->epilogue == Q3_GEMM_SWIGLU_BWD;
  if (d->epilogue < 0 || d->epilogue > Q3_GEMM_SWIGLU_BWD) return false;
  if (gate_up && (c.at || c.bt)) return false;
  if (sbwd && (c.at || !c.bt)) return false;
  if ((gate_up || sbwd) && a.axis != 0) return false;
  if (a.axis == 1 && !(c.bt && !c.at)) return false;
  if (a.axis == 2 && (c.at || c.bt)) return false;
  if (a.axis == 3 && !(c.at && c.bt)) return false;
  a.N = gate_up ? 2 * d->n : d->n;
  c.epi = gate_up ? 3 : sbwd ? 5 : 0;
  const int64_t total = a.axis == 1 ? d->k : a.axis == 2 ? d->n : d->m;
  int64_t beg = 0;
  for (int i = 0; i < 3; ++i) {
    if (i >= d->pieces) continue;
    const int64_t end = a.axis == 0 ? total : d->end[i], len = end - beg;
    if (len < 1 || end > total || (i + 1 == d->pieces && end != total)) return false;
    const int64_t pm = a.axis == 3 ? len : d->m, pn = a.axis == 2 ? len : d->n, pk = a.axis == 1 ? len : d->k;
    const int ia = a.axis == 2 ? 0 : i, ib = a.axis == 3 ? 0 : i, ic = a.axis == 1 ? 0 : i;
    if (!operand_ok(d->a[ia], d->lda[ia], pm, pk, c.at) || !operand_ok(d->b[ib], d->ldb[ib], pn, pk, c.bt)) return false;
    if (!d->c[ic] || d->ldc[ic] < pn) return false;
    a.len[i] = len;
    beg = end;
  }
  bool vec = d->n % 8 == 0;
  for (int i = 0; i < 3; ++i) {
    a.a.p[i] = (const u16*)d->a[i];
    a.a.ld[i] = d->lda[i];
    a.b.p[i] = (const u16*)d->b[i];
    a.b.ld[i] = d->ldb[i];
    a.c[i] = d->c[i];
    a.ldc[i] = d->ldc[i];
    if (i < d->pieces && a.axis >= 2) vec = vec && al16(d->c[i]) && d->ldc[i] % 8 == 0 && (a.axis == 3 || a.len[i] % 8 == 0);
  }
  vec = vec && al16(d->c[0]) && d->ldc[0] % 8 == 0;
  if (d->epilogue == Q3_GEMM_RESIDUAL || d->epilogue == Q3_GEMM_RESIDUAL_NORM) {
    if (a.axis != 0 || !d->res || d->ldres < d->n) return false;
    a.res = (const u16*)d->res;
    a.ldres = d->ldres;
    vec = vec && al16(d->res) && d->ldres % 8 == 0;
  }
  if (d->epilogue == Q3_GEMM_RESIDUAL_NORM &&
      !(vec && d->norm_w && d->y && al16(d->norm_w) && al16(d->y) && d->ldc[0] == d->n && d->ldy == d->n && d->n <= 8192 &&
        d->eps > 0.f))
    return false;
  if (gate_up) {
    if (!operand_ok(d->b[1], d->ldb[0], d->n, d->k, false) || !vec || !d->g != !d->u || !al16(d->g) || !al16(d->u))
      return false;
    a.g = (u16*)d->g;
    a.u = (u16*)d->u;
  }
  if (sbwd) {
    if (!vec || !d->c[1] || !al16(d->c[1]) || !d->g || !d->u || !al16(d->g) || !al16(d->u) || d->ldgu % 8 != 0 || d->ldgu < d->n)
      return false;
    a.gin = (const u16*)d->g;
    a.uin = (const u16*)d->u;
    a.ldgu = d->ldgu;
  }
  a.vec = vec;
  c.can_split = c.epi == 0 && vec;
  c.combine = d->epilogue == Q3_GEMM_RESIDUAL_NORM ? 0.5 : 4.5;
  // the smallest tiles, times the most splits, still number fewer than 2^31
  return tile_rows(a, 32) * tile_cols(a, 64) < (1ll << 28);
}

// One launch of a call: its arguments (the rows it forms are rows of its own operands), tiles and grid.
struct Launch {
  Args a;
  Plan p;
  int64_t rows;
};

void set_grid(Launch& l) {
  const Cfg& f = kCfg[l.p.cfg];
  l.a.tms = (int)(l.rows < l.a.M ? l.rows / f.bm : tile_rows(l.a, f.bm));
  l.a.tns = (int)tile_cols(l.a, f.bn);
}

int launch(const Call& c, const Launch& l, int dtype, hipStream_t s) {
  if (c.at) return q3gemm::launch_tile_tn(dtype, l.p.cfg, l.a, s);
  if (c.bt) return q3gemm::launch_tile_nn(dtype, l.p.cfg, c.epi, l.a, s);
  return q3gemm::launch_tile_nt(dtype, l.p.cfg, c.epi, l.a, s);
}

// 256 x 256 tiles whose last round leaves at least 3/8 of the CUs idle: the rows that fill whole rounds first,
// the rest as their own plan in a second launch (6144 x 4096 x 8192: 300 us against 333 us in one launch; the
// same per-element k order, so the same bits).
int64_t whole_round_rows(const Call& c, const Plan& p) {
  if (p.cfg != 0 || p.splits != 1) return 0;
  for (int i = 0; c.a.axis == 3 && i + 1 < c.a.pieces; ++i)
    if (c.a.len[i] % 256 != 0) return 0;
  const int64_t tn = tile_cols(c.a, 256), tiles = tile_rows(c.a, 256) * tn, rem = tiles % 256;
  if (tiles < 256 || rem == 0 || rem > 160 || 256 % tn != 0) return 0;
  return tiles / 256 * 256 / tn * 256;
}

// The call without its first rows: a call of its own, so that its tiles start at the first row left whatever
// their height, and no row is formed twice (the residual may be the output itself).
void drop_rows(Args& a, bool at, int64_t rows) {
  a.M -= rows;
  if (a.axis == 3) {
    for (; rows >= a.len[0]; --a.pieces) {
      rows -= a.len[0];
      for (int i = 0; i + 1 < a.pieces; ++i) {
        a.a.p[i] = a.a.p[i + 1];
        a.a.ld[i] = a.a.ld[i + 1];
        a.c[i] = a.c[i + 1];
        a.ldc[i] = a.ldc[i + 1];
        a.len[i] = a.len[i + 1];
      }
    }
    a.len[0] -= rows;
  }
  for (int i = 0; i < (a.axis == 1 ? a.pieces : 1); ++i) a.a.p[i] += at ? rows : rows * a.a.ld[i];
  for (int i = 0; i < (a.axis == 3 ? 1 : 3); ++i)  // axis 2: every piece; dg and du share dg's stride
    if (a.c[i]) a.c[i] = (u16*)a.c[i] + rows * a.ldc[a.axis == 2 ? i : 0];
  const int64_t out = rows * a.ldc[0], in = rows * a.ldgu;
  if (a.res) a.res += rows * a.ldres;
  if (a.g) a.g += out;
  if (a.u) a.u += out;
  if (a.gin) a.gin += in;
  if (a.uin) a.uin += in;
}

// The launches of a call, one or two.
int launches(const Call& c, Launch* l) {
  l[0].a = c.a;
  l[0].p = plan_for(c.a, c.at, c.bt, c.can_split, c.combine);
  l[0].a.splits = l[0].p.splits;
  const int64_t m1 = whole_round_rows(c, l[0].p);
  l[0].rows = m1 > 0 ? m1 : c.a.M;
  set_grid(l[0]);
  if (m1 == 0) return 1;
  l[1].a = c.a;
  drop_rows(l[1].a, c.at, m1);
  l[1].p = plan_for(l[1].a, c.at, c.bt, false, c.combine);
  l[1].rows = l[1].a.M;
  set_grid(l[1]);
  return 2;
}

}  // namespace

extern "C" {

size_t q3_gemm_workspace_bytes(const q3_gemm_desc* d) {
  Call c;
  if (!parse(d, c)) return 0;
  const Plan p = plan_for(c.a, c.at, c.bt, c.can_split, c.combine);
  return p.splits > 1 ? (size_t)p.splits * (size_t)c.a.M * (size_t)c.a.N * sizeof(float) : 0;
}

int q3_gemm_plan(const q3_gemm_desc* d, int64_t* out) {
  Call c;
  Launch l[2];
  if (!out || !parse(d, c)) return 0;
  const int n = launches(c, l);
  for (int i = 0; i < n; ++i) {
    const Cfg& f = kCfg[l[i].p.cfg];
    const int64_t row[5] = {c.a.M - l[i].a.M, l[i].rows, f.bm, f.bn, l[i].p.splits};
    std::copy(row, row + 5, out + 5 * i);
  }
  return n;
}

int q3_gemm(const q3_gemm_desc* d, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  Call c;
  Q3_REQUIRE(parse(d, c));
  Launch l[2];
  const int n = launches(c, l);
  const bool norm = d->epilogue == Q3_GEMM_RESIDUAL_NORM;
  if (l[0].p.splits > 1) {
    Args& a = l[0].a;
    Q3_REQUIRE(workspace && al16(workspace) &&
               workspace_bytes >= (size_t)a.splits * (size_t)a.M * (size_t)a.N * sizeof(float));
    a.part = (float*)workspace;
    const int rc = launch(c, l[0], d->dtype, stream);
    if (rc != 0) return rc;
    if (norm) {
      if (d->dtype == Q3_BF16)
        combine_norm_kernel<BF16><<<(unsigned)a.M, 512, 0, stream>>>(a, (const u16*)d->norm_w, d->eps, (u16*)d->y, d->ldy);
      else
        combine_norm_kernel<F16><<<(unsigned)a.M, 512, 0, stream>>>(a, (const u16*)d->norm_w, d->eps, (u16*)d->y, d->ldy);
    } else {
      const unsigned g = (unsigned)cdiv(a.M * (a.N / 8), 256);
      if (d->dtype == Q3_BF16) combine_kernel<BF16><<<g, 256, 0, stream>>>(a);
      else combine_kernel<F16><<<g, 256, 0, stream>>>(a);
    }
    return (int)hipGetLastError();
  }
  for (int i = 0; i < n; ++i) {
    const int rc = launch(c, l[i], d->dtype, stream);
    if (rc != 0) return rc;
  }
  return norm ? q3_rmsnorm_fwd(d->dtype, d->c[0], d->norm_w, d->y, d->m, d->n, d->eps, stream) : 0;
}

// LM-head logits A B^T, stored, with their cross-entropy statistics (q3hip.h): 256 x 256 tiles, 128 x 256 when
// those would leave half of the last (or only) row of tiles empty.
int q3_gemm_nt_ce_stats_store(int dtype, const void* A, int64_t lda, const void* B, int64_t ldb, int64_t M, int64_t N,
                              int64_t K, int64_t col0, const int64_t* tgt, float* m_part, float* s_part, float* pick,
                              int64_t part0, int64_t ldp, void* z, int64_t ldz, hipStream_t stream) {
  Q3_REQUIRE((dtype == Q3_BF16 || dtype == Q3_F16) && tgt && m_part && s_part && pick);
  Q3_REQUIRE(M > 0 && N > 0 && K > 0 && M < (1ll << 31) - 256 && N < (1ll << 30) && K < (1ll << 31) && K % 64 == 0);
  Q3_REQUIRE(operand_ok(A, lda, M, K, false) && operand_ok(B, ldb, N, K, false) && ldp >= M && part0 >= 0);
  Q3_REQUIRE(z && ldz >= N && ldz % 8 == 0 && al16(z));
  Args a{};
  a.a.p[0] = (const u16*)A;
  a.a.ld[0] = lda;
  a.b.p[0] = (const u16*)B;
  a.b.ld[0] = ldb;
  a.M = M;
  a.N = N;
  a.K = K;
  a.pieces = a.splits = 1;
  a.c[0] = z;
  a.ldc[0] = ldz;
  a.tgt = tgt;
  a.m_part = m_part;
  a.s_part = s_part;
  a.pick = pick;
  a.part0 = part0;
  a.ldp = ldp;
  a.col0 = col0;
  const bool big = M > 128 && (M % 256 == 0 || M % 256 > 128 || M > 2048);
  a.tms = (int)cdiv(M, big ? 256 : 128);
  a.tns = (int)cdiv(N, 256);
  Q3_REQUIRE((int64_t)a.tms * a.tns < (1ll << 31));
  return q3gemm::launch_tile_nt(dtype, big ? 0 : 1, 2, a, stream);
}

}  // extern "C"
