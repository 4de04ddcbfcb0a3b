// The three products of the gate/up projection's backward in one launch:
//   dx      = da W_gate + db W_up          [M, D]   (K = 2 H)
//   dW_gate = da^T x,  dW_up = db^T x      [H, D]   (K = the M tokens)
// (the Linears' gradients in the reference's SwiGLUMLP backward,
// model/dit.py:104-110), from da, db, x and the weights as they lie in memory.
//
// Every output row is D long and contiguous, so the products are formed
// transposed, tiles of 256 (D) x 256 (tokens or hidden units): the A operand
// is W or x read M-major (D contiguous, transposing LDS reads), B is da / db,
// K-contiguous for dx and N-major for dW.  A lane then holds 4 consecutive
// elements of an output row per 32x32 tile quarter, and one exchange between
// the lane halves makes 16-byte stores.  Nothing is transposed through memory
// (the transposes of da, db and x that a K-contiguous weight product needs
// took 26 us of the encoder MLP's backward, 42 us at M 4096 D 2048 H 5632),
// dx's two terms add in fp32, and the long dx tiles and the dW tiles fill the
// chip together.
//
// Each product may be split along K into S fp32 slices added in order by
// gate_up_reduce_kernel; pick_split picks the splits.  Large bf16 products keep
// the earlier form: nf_gemm_swiglu_bwd_wins.
#include "gemm_store.h"

namespace nf {
namespace gate_up {

using C = gemm::DCfg<256, 256, 2, 4, 2, 64>;
using gemm::floatx16;
using OpK = gemm::DtlOperandKN<C>;

// One of the launch's three products.
struct Job {
  void *out;      // [rows, D], null: not wanted
  float *part;    // [S, rows, D] fp32 when S > 1
  int64_t rows;   // output rows: tokens (dx) or hidden units (dW)
  int dt;         // element type of out
  int tiles_n;    // 256-row tiles
  int blocks;     // tiles_d * tiles_n * S, 0 when not wanted
  int S;
  int stages;     // 64-deep K stages per slice
};

struct Args {
  const bf16 *da, *db, *x, *wg, *wu;
  int64_t ld_ab, ldx, ldg, ldu, M, D, H;
  int tiles_d;
  int first_w;    // the dW blocks come before the dx blocks
  Job dx, dwg, dwu;
};

// Rows n of the output, columns m: element (m, n) of the tile's product goes to
// out[n * D + m].  VEC: D a multiple of 8 and out 16-byte aligned.
template <bool VEC>
__device__ __forceinline__ void store_rows(const floatx16 (&acc)[C::TM][C::TN], void *out, int dt,
                                           int64_t D, int64_t rows, int64_t m0, int64_t n0) {
  const int l = threadIdx.x & 63, half = l >> 5;
  const int w = threadIdx.x >> 6, wm = w / C::WN, wn = w % C::WN;
#pragma unroll
  for (int j = 0; j < C::TN; ++j) {
    const int64_t n = n0 + wn * C::WTN + j * 32 + (l & 31);
#pragma unroll
    for (int i = 0; i < C::TM; ++i) {
      const int64_t mt = m0 + wm * C::WTM + i * 32;
      if constexpr (!VEC) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t m = mt + 8 * (r >> 2) + 4 * half + (r & 3);
          if (n < rows && m < D) store_dyn(out, dt, n * D + m, acc[i][j][r]);
        }
      } else if (dt == NF_DTYPE_F32) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int64_t m = mt + 8 * g + 4 * half;
          u32x4 v;
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = __float_as_uint(acc[i][j][4 * g + q]);
          if (n < rows && m < D)
            *reinterpret_cast<u32x4 *>(static_cast<float *>(out) + n * D + m) = v;
        }
      } else {
        // quarters g and g + 1: the swap leaves lanes 0-31 with all of g,
        // lanes 32-63 with all of g + 1
#pragma unroll
        for (int g = 0; g < 4; g += 2) {
          uint32_t a[2], b[2];
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            a[q] = (uint32_t)gemm::to_half_bits(acc[i][j][4 * g + 2 * q], dt) |
                   ((uint32_t)gemm::to_half_bits(acc[i][j][4 * g + 2 * q + 1], dt) << 16);
            b[q] = (uint32_t)gemm::to_half_bits(acc[i][j][4 * g + 4 + 2 * q], dt) |
                   ((uint32_t)gemm::to_half_bits(acc[i][j][4 * g + 5 + 2 * q], dt) << 16);
          }
          const auto s0 = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
          const auto s1 = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
          const u32x4 v = {s0[0], s1[0], s0[1], s1[1]};
          const int64_t m = mt + 8 * (g + half);
          if (n < rows && m < D)
            *reinterpret_cast<u32x4 *>(static_cast<uint16_t *>(out) + n * D + m) = v;
        }
      }
    }
  }
}

template <bool BUF>
__device__ __forceinline__ void finish(const floatx16 (&acc)[C::TM][C::TN], const Job &jb, int s,
                                       int64_t D, int64_t m0, int64_t n0) {
  if (jb.S > 1)
    store_rows<BUF>(acc, jb.part + (int64_t)s * jb.rows * D, NF_DTYPE_F32, D, jb.rows, m0, n0);
  else
    store_rows<BUF>(acc, jb.out, jb.dt, D, jb.rows, m0, n0);
}

__device__ __forceinline__ void clear(floatx16 (&acc)[C::TM][C::TN]) {
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
}

// BUF: rows of whole 16-byte vectors (D, H and the strides multiples of 8,
// aligned bases): buffer copies and vector stores; else (views of other
// alignments, padded rows past 2 GiB) register copies and element stores.
template <bool BUF>
__global__ NF_GEMM_BOUNDS(C) void gate_up_bwd_kernel(Args p) {
  __shared__ __attribute__((aligned(16))) char smem[C::LDS_BYTES];
  const int nw = p.dwg.blocks + p.dwu.blocks;
  int b = (int)blockIdx.x;
  const bool is_w = p.first_w ? b < nw : b >= p.dx.blocks;
  b -= is_w ? (p.first_w ? 0 : p.dx.blocks) : (p.first_w ? nw : 0);
  const bool up = is_w && b >= p.dwg.blocks;
  if (up) b -= p.dwg.blocks;
  const Job &jb = is_w ? (up ? p.dwu : p.dwg) : p.dx;
  const int t = gemm::xcd_order(b, jb.blocks);
  const int per = p.tiles_d * jb.tiles_n;
  const int s = t / per;  // K slice
  int td, tn;
  gemm::group_tile(t % per, p.tiles_d, jb.tiles_n, gemm::kTileGroup, td, tn);
  const int64_t m0 = (int64_t)td * C::BM, n0 = (int64_t)tn * C::BN;
  const int64_t k0 = (int64_t)s * jb.stages * C::BK;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  floatx16 acc[C::TM][C::TN];
  clear(acc);
  OpK opa;
  if (is_w) {  // K: the tokens
    const int64_t left = p.M - k0, kl = (int64_t)jb.stages * C::BK;
    const int64_t klen = left < kl ? (left < 0 ? 0 : left) : kl;
    OpK opb;
    opa.init(p.x + k0 * p.ldx, p.ldx, p.D, klen, m0, wave);
    opb.init((up ? p.db : p.da) + k0 * p.ld_ab, p.ld_ab, p.H, klen, n0, wave);
    gemm::mainloop_dtl_ops<C, BUF, true>(opa, opb, klen, smem, acc);
    finish<BUF>(acc, jb, s, p.D, m0, n0);
  } else {  // K: the gate units, then the up units, each padded to whole stages
    const int64_t hs = (p.H + C::BK - 1) / C::BK * C::BK, k1 = k0 + (int64_t)jb.stages * C::BK;
#pragma unroll 1
    for (int seg = 0; seg < 2; ++seg) {
      const int64_t lo = (k0 > seg * hs ? k0 : seg * hs) - seg * hs;
      int64_t hi = (k1 < (seg + 1) * hs ? k1 : (seg + 1) * hs) - seg * hs;
      if (hi > p.H) hi = p.H;
      if (lo >= hi) continue;
      const int64_t ldw = seg ? p.ldu : p.ldg;
      gemm::DtlOperand<C, C::BCW> opb;
      opa.init((seg ? p.wu : p.wg) + lo * ldw, ldw, p.D, hi - lo, m0, wave);
      opb.init((seg ? p.db : p.da) + lo, p.ld_ab, p.M, hi - lo, n0, wave);
      gemm::mainloop_dtl_ops<C, BUF, false>(opa, opb, hi - lo, smem, acc);
    }
    finish<BUF>(acc, jb, s, p.D, m0, n0);
  }
}

// out[i] = the sum of the job's S slices at i, in slice order; up to three
// jobs, each over blocks of its own.  4 elements per thread when VEC.
struct Sum {
  const float *part;
  void *out;
  int64_t n;   // elements
  int S, dt;
  int blocks;  // 0: none
};
struct Sums {
  Sum j[3];
};
constexpr int kSumThreads = 256;
template <bool VEC>
__global__ __launch_bounds__(kSumThreads) void gate_up_reduce_kernel(Sums p) {
  int b = (int)blockIdx.x, k = 0;
  while (k < 2 && b >= p.j[k].blocks) b -= p.j[k++].blocks;
  const Sum &q = p.j[k];
  constexpr int VE = VEC ? 4 : 1;
  for (int64_t i = ((int64_t)b * kSumThreads + threadIdx.x) * VE; i < q.n;
       i += (int64_t)q.blocks * kSumThreads * VE) {
    float a[VE];
#pragma unroll
    for (int e = 0; e < VE; ++e) a[e] = 0.f;
    constexpr int kBatch = 8;
    for (int s0 = 0; s0 < q.S; s0 += kBatch) {
      float v[kBatch][VE];
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (s0 + u < q.S) __builtin_memcpy(v[u], q.part + (s0 + u) * q.n + i, sizeof(v[u]));
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (s0 + u < q.S)
#pragma unroll
          for (int e = 0; e < VE; ++e) a[e] += v[u][e];
    }
    if constexpr (VEC) {
      if (q.dt == NF_DTYPE_F32) {
        *reinterpret_cast<float4 *>(static_cast<float *>(q.out) + i) =
            make_float4(a[0], a[1], a[2], a[3]);
      } else {
        u32x2 h;
        h.x = gemm::to_half_bits(a[0], q.dt) | ((uint32_t)gemm::to_half_bits(a[1], q.dt) << 16);
        h.y = gemm::to_half_bits(a[2], q.dt) | ((uint32_t)gemm::to_half_bits(a[3], q.dt) << 16);
        *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(q.out) + i) = h;
      }
    } else {
      store_dyn(q.out, q.dt, i, a[0]);
    }
  }
}

// Rows that are not whole 16-byte vectors (D or H no multiple of 8): each tile would
// read them two bytes at a time through registers.  So the operands are copied
// once to rows of Dp and Hp elements, zeros past D and H, the products run on Dp
// and Hp, into fp32 slices, and the reduce below drops the padding.  Forward +
// backward, us, element-wise tiles -> padded: M 9408 D 383 H 1537 482 -> 274, M
// 4096 D 2047 H 5631 2446 -> 1308, M 300 D 77 H 501 71 -> 45, M 64 D 300 H 1030
// 75 -> 58.  Up to five matrices a launch; a block takes kSumThreads vectors of one.
struct Pad {
  const bf16 *in;
  bf16 *out;
  int64_t rows, cols, ld;  // what is there
  int64_t ld_out;          // elements a padded row
  int64_t vectors, blocks; // of the padded rows
};
struct Pads {
  Pad j[5];
  int n;
};
static __global__ __launch_bounds__(kSumThreads) void gate_up_pad_kernel(Pads p) {
  int64_t b = blockIdx.x;
  int k = 0;
  while (k < p.n - 1 && b >= p.j[k].blocks) b -= p.j[k++].blocks;
  const Pad &q = p.j[k];
  const int64_t v = b * kSumThreads + threadIdx.x;
  if (v >= q.vectors) return;
  const int64_t vpr = q.ld_out / 8, r = v / vpr, c = (v - r * vpr) * 8;
  const bf16 *src = q.in + r * q.ld + c;
  bf16 e[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    e[i] = r < q.rows && c + i < q.cols ? src[i] : static_cast<bf16>(0.f);
  u32x4 w;
  __builtin_memcpy(&w, e, 16);
  *reinterpret_cast<u32x4 *>(q.out + v * 8) = w;
}

// out[r, c] = the sum of the S slices at (r, c) of their rows of `pitch`, r < rows,
// c < cols; up to three products, as above.
struct PadSum {
  const float *part;
  void *out;
  int64_t rows, cols, pitch, slice;
  int S, dt;
  int64_t blocks;
};
struct PadSums {
  PadSum j[3];
  int n;
};
static __global__ __launch_bounds__(kSumThreads) void gate_up_pad_reduce_kernel(PadSums p) {
  int64_t b = blockIdx.x;
  int k = 0;
  while (k < p.n - 1 && b >= p.j[k].blocks) b -= p.j[k++].blocks;
  const PadSum &q = p.j[k];
  const int64_t v = b * kSumThreads + threadIdx.x, vpr = q.pitch / 4;
  const int64_t r = v / vpr, c = (v - r * vpr) * 4;
  if (r >= q.rows) return;
  float a[4] = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < q.S; ++s) {
    const float4 x = *reinterpret_cast<const float4 *>(q.part + s * q.slice + v * 4);
    a[0] += x.x; a[1] += x.y; a[2] += x.z; a[3] += x.w;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (c + i < q.cols) store_dyn(q.out, q.dt, r * q.cols + c + i, a[i]);
}

// K splits of the launch.  nx dx tiles of kx stages and nw dW tiles of kw
// stages run on 256 CUs, one block each, the longer blocks first; a block
// also costs ~4 stages of prologue and epilogue, and a split product the
// write and read of its fp32 slices (stages of ~1.8 us against ~5 TB/s).  A few
// tokens against a wide H leave one or two dx tiles of all K: M 48 D 256 H 11008,
// forward + backward, 103 us with at most 8 dx slices, 55 with up to 32.
struct Split {
  int sx, sw;
};
inline Split pick_split(int64_t M, int64_t D, int64_t H, bool want_x, int want_w) {
  const int64_t td = (D + C::BM - 1) / C::BM;
  const int64_t nx = want_x ? td * ((M + C::BN - 1) / C::BN) : 0;
  const int64_t nw = want_w * td * ((H + C::BN - 1) / C::BN);
  const int64_t kx = 2 * ((H + C::BK - 1) / C::BK), kw = (M + C::BK - 1) / C::BK;
  const double over = 4.0, per_byte = 1.0 / (5e12 * 1.8e-6);
  Split best{1, 1};
  double best_t = -1.0;
  for (int sx = 1; sx <= 32 && (sx == 1 || (want_x && kx / sx >= 4)); sx += sx < 8 ? 1 : sx / 4)
    for (int sw = 1; sw <= 32 && (sw == 1 || (want_w && kw / sw >= 4)); ++sw) {
      const double lx = (double)((kx + sx - 1) / sx) + over, lw = (double)((kw + sw - 1) / sw) + over;
      double t = lx >= lw ? gemm::two_job_makespan(nx * sx, lx, nw * sw, lw)
                          : gemm::two_job_makespan(nw * sw, lw, nx * sx, lx);
      if (sx > 1) t += 2.0 * sx * (double)M * D * 4 * per_byte;
      if (sw > 1) t += 2.0 * sw * want_w * (double)H * D * 4 * per_byte;
      if (best_t < 0 || t < best_t * 0.999) {
        best_t = t;
        best = {sx, sw};
      }
    }
  return best;
}

// rows x ld elements of 2 bytes stay under 2 GiB (32-bit buffer offsets)
inline bool under_2gib(int64_t rows, int64_t ld) {
  const int64_t lim = (((int64_t)1 << 31) - 64) / 2;
  return rows >= 0 && ld > 0 && ld <= lim && rows <= (lim - 1) / ld;
}

struct Layout {
  Split sp;
  bool pad;        // the products run on padded copies, rows of Dp and Hp
  int64_t Dp, Hp;  // D and H where not
  size_t off_x, off_g, off_u;  // the products' slices
  size_t off_da, off_db, off_xp, off_wg, off_wu;  // the copies
  size_t total;
};
// A thread keeps its last shape's layout: the workspace call and the launch
// of every step ask for the same one.
inline Layout layout(int64_t M, int64_t D, int64_t H, bool x, bool g, bool u) {
  struct Kept {
    int64_t M, D, H;
    int want;
    Layout L;
  };
  static thread_local Kept kept{0, 0, 0, 0, {}};
  const int want = (int)x + 2 * (int)g + 4 * (int)u;
  if (kept.M == M && kept.D == D && kept.H == H && kept.want == want) return kept.L;
  Layout L{};
  const int64_t dp = gemm::round_up(D, 8), hp = gemm::round_up(H, 8);
  L.pad = (dp != D || hp != H) && under_2gib(M, dp) && under_2gib(M, hp) && under_2gib(hp, dp);
  L.Dp = L.pad ? dp : D;
  L.Hp = L.pad ? hp : H;
  L.sp = pick_split(M, L.Dp, L.Hp, x, (int)g + (int)u);
  size_t o = 0;
  auto take = [&](size_t bytes) { const size_t at = o; o = gemm::align256(o + bytes); return at; };
  auto slices = [&](bool want, int S, int64_t rows) {
    return take(want && (S > 1 || L.pad) ? (size_t)S * rows * L.Dp * sizeof(float) : 0);
  };
  auto copy = [&](bool want, int64_t rows, int64_t cols) {
    return take(L.pad && want ? (size_t)rows * cols * sizeof(bf16) : 0);
  };
  L.off_x = slices(x, L.sp.sx, M);
  L.off_g = slices(g, L.sp.sw, L.Hp);
  L.off_u = slices(u, L.sp.sw, L.Hp);
  L.off_da = copy(x || g, M, L.Hp);
  L.off_db = copy(x || u, M, L.Hp);
  L.off_xp = copy(g || u, M, L.Dp);
  L.off_wg = copy(x, L.Hp, L.Dp);
  L.off_wu = copy(x, L.Hp, L.Dp);
  L.total = o;
  kept = {M, D, H, want, L};
  return L;
}

// The launch on padded copies: a holds the padded extents and the operands as they
// lie, its jobs' slices the padded products.
inline int launch_padded(Args a, const Layout &L, char *ws, int64_t total, void *dx, int dt_dx,
                         void *dw_gate, void *dw_up, int dt_dw, int64_t D, int64_t H,
                         hipStream_t s) {
  const bool any_w = dw_gate || dw_up;
  Pads pd{};
  int64_t blocks = 0;
  auto pad = [&](const bf16 *&m, size_t off, int64_t rows, int64_t cols, int64_t ld,
                 int64_t rows_out, int64_t ld_out) {
    bf16 *out = reinterpret_cast<bf16 *>(ws + off);
    const int64_t vectors = rows_out * (ld_out / 8);
    const int64_t nb = (vectors + kSumThreads - 1) / kSumThreads;
    pd.j[pd.n++] = Pad{m, out, rows, cols, ld, ld_out, vectors, nb};
    blocks += nb;
    m = out;
  };
  if (dx || dw_gate) pad(a.da, L.off_da, a.M, H, a.ld_ab, a.M, L.Hp);
  if (dx || dw_up) pad(a.db, L.off_db, a.M, H, a.ld_ab, a.M, L.Hp);
  if (any_w) pad(a.x, L.off_xp, a.M, D, a.ldx, a.M, L.Dp);
  if (dx) pad(a.wg, L.off_wg, H, D, a.ldg, L.Hp, L.Dp);
  if (dx) pad(a.wu, L.off_wu, H, D, a.ldu, L.Hp, L.Dp);
  a.ld_ab = L.Hp;
  a.ldx = a.ldg = a.ldu = L.Dp;
  PadSums q{};
  int64_t sum_blocks = 0;
  auto sum = [&](const Job &j, void *out, int64_t rows, int dt) {
    if (!out) return;
    const int64_t nb = (rows * (L.Dp / 4) + kSumThreads - 1) / kSumThreads;
    q.j[q.n++] = PadSum{j.part, out, rows, D, L.Dp, j.rows * L.Dp, j.S, dt, nb};
    sum_blocks += nb;
  };
  sum(a.dx, dx, a.M, dt_dx);
  sum(a.dwg, dw_gate, H, dt_dw);
  sum(a.dwu, dw_up, H, dt_dw);
  if (blocks > 0x7fffffffLL || sum_blocks > 0x7fffffffLL)
    return set_error(NF_ERR_ARG, "nf_gemm_swiglu_bwd: grid too large");
  gate_up_pad_kernel<<<(unsigned)blocks, kSumThreads, 0, s>>>(pd);
  if (int e = check_launch("gate_up_pad")) return e;
  gate_up_bwd_kernel<true><<<(unsigned)total, C::NT, 0, s>>>(a);
  if (int e = check_launch("nf_gemm_swiglu_bwd")) return e;
  gate_up_pad_reduce_kernel<<<(unsigned)sum_blocks, kSumThreads, 0, s>>>(q);
  return check_launch("gate_up_pad_reduce");
}

}  // namespace gate_up
}  // namespace nf

using namespace nf;

// The line between the one launch and what it stands beside for bf16 (dx as two
// library GEMMs, nf_gemm_swiglu_wgrad on transposed copies, dx's two terms
// rounded in between).  The M- and N-major operands take twice the LDS reads of
// K-contiguous ones, which costs more than transposing once the products are
// long in all three extents and power-bound.  Forward + backward, us, one launch
// against the other form:
//   M 4096 D 2048 H 5632 627 / 656;   M 2048 D 3072 H 8192 665 / 668;
//   M 8192 D 1536 H 8192 1336 / 1357; M 65536 D 2048 H 1536 2649 / 2779;
//   M 4096 D 5120 H 2736 756 / 836;   M 1024 D 4096 H 11008 668 / 682;
//   M 4096 D 3072 H 5632 912 / 898;   M 4096 D 2048 H 11008 1284 / 1190;
//   M 8192 D 2048 H 5632 1302 / 1208; M 4096 D 4096 H 11008 2270 / 1970;
//   M 16384 D 4096 H 5632 4398 / 3880; M 8192 D 8192 H 8192 5996 / 5202.
// (The transposed copies, M padded to 8, must stay under 2 GiB.)
// dx alone (frozen weights) has no transposes to weigh against, so the library's
// products win sooner: M 9408 D 1000 H 2731 439 / 358, M 9408 D 384 H 1536 120 / 111,
// M 16384 D 1536 H 4096 1042 / 904, M 4096 D 2048 H 5632 447 / 411; M 4096 D 768 H
// 3072 144 / 153, M 2048 D 1536 H 4096 145 / 162, M 512 D 2048 H 5632 113 / 129.
extern "C" int nf_gemm_swiglu_bwd_wins(int64_t M, int64_t D, int64_t H, int want_dw) {
  const double work = (double)M * (double)D * (double)H;
  if (!want_dw) return !(M >= 8192 || work >= 2.5e10);
  const bool large = M >= 2048 && D >= 2048 && H >= 2560 && work >= 6.5e10;
  return !(large && gate_up::under_2gib(M + 7, H > D ? H : D));
}

extern "C" size_t nf_gemm_swiglu_bwd_workspace(int64_t M, int64_t D, int64_t H, int want_dx,
                                               int want_dgate, int want_dup) {
  const int64_t big = (int64_t)1 << 31;
  if (M <= 0 || D <= 0 || H <= 0 || M > big || D > big || H > big) return 0;
  return gate_up::layout(M, D, H, want_dx, want_dgate, want_dup).total;
}

extern "C" int nf_gemm_swiglu_bwd(const void *da, const void *db, int64_t ld_ab, const void *x,
                                  int64_t ldx, const void *w_gate, int64_t ld_gate,
                                  const void *w_up, int64_t ld_up, void *dx, int dt_dx,
                                  void *dw_gate, void *dw_up, int dt_dw, int64_t M, int64_t D,
                                  int64_t H, int dtype, void *workspace, size_t workspace_bytes,
                                  void *stream) {
  using namespace nf::gate_up;
  if (M < 0 || D <= 0 || H <= 0)
    return set_error(NF_ERR_ARG, "nf_gemm_swiglu_bwd: bad shape M=%lld D=%lld H=%lld",
                     (long long)M, (long long)D, (long long)H);
  if (dtype != NF_DTYPE_BF16)
    return set_error(NF_ERR_DTYPE, "nf_gemm_swiglu_bwd: dtype %d unsupported (bf16 only)", dtype);
  if (!is_dtype(dt_dx) || !is_dtype(dt_dw))
    return set_error(NF_ERR_DTYPE, "nf_gemm_swiglu_bwd: gradient dtypes %d, %d", dt_dx, dt_dw);
  const bool any_w = dw_gate || dw_up;
  if (M > 0 && (!da || !db || (any_w && !x) || (dx && (!w_gate || !w_up))))
    return set_error(NF_ERR_ARG, "nf_gemm_swiglu_bwd: null pointer");
  if (ld_ab < H || ldx < D || ld_gate < D || ld_up < D)
    return set_error(NF_ERR_ARG, "nf_gemm_swiglu_bwd: bad leading dimension");
  if (!under_2gib(M, ld_ab) || !under_2gib(M, ldx) || !under_2gib(H, ld_gate) ||
      !under_2gib(H, ld_up))
    return set_error(NF_ERR_ARG, "nf_gemm_swiglu_bwd: an operand exceeds 2 GiB");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (M == 0) {  // no tokens: zero weight gradients
    const int64_t cols = D * (dt_dw == NF_DTYPE_F32 ? 2 : 1);  // 16-bit elements
    for (void *w : {dw_gate, dw_up})
      if (w)
        if (int e = gemm::launch_zero16(w, cols, H, cols, s)) return e;
    return NF_OK;
  }
  if (!dx && !any_w) return NF_OK;
  const Layout L = layout(M, D, H, dx, dw_gate, dw_up);
  if (L.total > 0 && (!workspace || workspace_bytes < L.total || !aligned16(workspace)))
    return set_error(NF_ERR_WORKSPACE, "nf_gemm_swiglu_bwd: workspace %zu bytes < required %zu",
                     workspace_bytes, L.total);
  char *ws = static_cast<char *>(workspace);
  Args a{};
  a.da = static_cast<const bf16 *>(da);
  a.db = static_cast<const bf16 *>(db);
  a.x = static_cast<const bf16 *>(x);
  a.wg = static_cast<const bf16 *>(w_gate);
  a.wu = static_cast<const bf16 *>(w_up);
  a.ld_ab = ld_ab; a.ldx = ldx; a.ldg = ld_gate; a.ldu = ld_up;
  a.M = M; a.D = L.Dp; a.H = L.Hp;
  a.tiles_d = (int)((a.D + C::BM - 1) / C::BM);
  int64_t total = 0;
  auto job = [&](void *out, size_t off, int64_t rows, int dt, int64_t K_stages, int S) {
    Job j{};
    j.out = out;
    j.part = reinterpret_cast<float *>(ws + off);
    j.rows = rows;
    j.dt = dt;
    j.tiles_n = (int)((rows + C::BN - 1) / C::BN);
    j.stages = (int)((K_stages + S - 1) / S);
    j.S = (int)((K_stages + j.stages - 1) / j.stages);
    if (L.pad && out && j.S == 1) {  // one slice: the sum's input all the same
      j.out = j.part;
      j.dt = NF_DTYPE_F32;
    }
    const int64_t blocks = out ? (int64_t)a.tiles_d * j.tiles_n * j.S : 0;
    total += blocks;
    j.blocks = (int)blocks;
    return j;
  };
  const int64_t kx = 2 * ((a.H + C::BK - 1) / C::BK), kw = (M + C::BK - 1) / C::BK;
  a.dx = job(dx, L.off_x, M, dt_dx, kx, L.sp.sx);
  a.dwg = job(dw_gate, L.off_g, a.H, dt_dw, kw, L.sp.sw);
  a.dwu = job(dw_up, L.off_u, a.H, dt_dw, kw, L.sp.sw);
  if (total > 0x7fffffffLL) return set_error(NF_ERR_ARG, "nf_gemm_swiglu_bwd: grid too large");
  a.first_w = a.dwg.stages > a.dx.stages;
  if (L.pad) return launch_padded(a, L, ws, total, dx, dt_dx, dw_gate, dw_up, dt_dw, D, H, s);
  const bool buf = D % 8 == 0 && H % 8 == 0 && ld_ab % 8 == 0 && ldx % 8 == 0 &&
                   ld_gate % 8 == 0 && ld_up % 8 == 0 && aligned16(da) && aligned16(db) &&
                   aligned16(x) && aligned16(w_gate) && aligned16(w_up) && aligned16(dx) &&
                   aligned16(dw_gate) && aligned16(dw_up);
  if (buf)
    gate_up_bwd_kernel<true><<<(unsigned)total, C::NT, 0, s>>>(a);
  else
    gate_up_bwd_kernel<false><<<(unsigned)total, C::NT, 0, s>>>(a);
  if (int e = check_launch("nf_gemm_swiglu_bwd")) return e;
  Sums q{};
  int nq = 0;
  unsigned blocks = 0;
  for (const Job *j : {&a.dx, &a.dwg, &a.dwu}) {
    if (!j->out || j->S <= 1) continue;
    const int64_t n = j->rows * D;
    int64_t nb = (n / (buf ? 4 : 1) + kSumThreads - 1) / kSumThreads;
    if (nb > 2048) nb = 2048;
    q.j[nq++] = Sum{j->part, j->out, n, j->S, j->dt, (int)nb};
    blocks += (unsigned)nb;
  }
  if (nq == 0) return NF_OK;
  if (buf)
    gate_up_reduce_kernel<true><<<blocks, kSumThreads, 0, s>>>(q);
  else
    gate_up_reduce_kernel<false><<<blocks, kSumThreads, 0, s>>>(q);
  return check_launch("gate_up_reduce");
}
