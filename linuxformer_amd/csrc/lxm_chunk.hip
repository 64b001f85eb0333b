// The stock forward's chunked delta rule (torch_chunk_gated_delta_rule, transformers qwen3_5
// :249-327) in chunks of <= 64 positions, on MI355X's matrix cores.
//
// Per (value head, chunk), with gc the cumulative sum of g and Gamma[i][j] = exp(gc_i - gc_j) for
// j <= i, else 0:
//   A2 = (q k^T) * Gamma;  L = (k beta k^T) * Gamma below the diagonal;  T = (I + L)^-1  (the
//   stock loop's result + I);  W = T (k beta exp(gc));  U = T (v beta)
//   v_new = U - W S;  o = (q exp(gc)) S + A2 v_new;  S <- S exp(g_last) + (k exp(g_last - gc))^T v_new
// A2, W and U need no state, so a sequence's chunks form them in parallel (chunk_prep, one
// workgroup per (head, chunk), into a workspace); what is left of a chunk is a short chain in the
// state (chunk_run, one workgroup per (head, 16 state columns), its chunks in order, the state
// in registers and LDS). One chunk alone (chunk_one) does both in one launch with no workspace.
//
// Every product is v_mfma_f32_16x16x4_f32 (a 16 x 16 tile += 16 x 4 times 4 x 16; lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16] and holds D[4 (l / 16) + r][l % 16], r = 0..3), its k
// ascending, so each result is one chain of fused multiply-adds in k order whatever the kernel.
// Operands come as 16 bytes a lane (a block of 16 k: lane group g's k = g, 4 + g, 8 + g, 12 + g):
// rows lie in LDS with each block of 16 transposed as 4 x 4 (pos16), tiles in LDS and in the
// workspace as operands, a D tile turned into a B operand by four 4-byte LDS writes a lane.
//
// A chunk's chain is bound by its latency: a wave's two products of 32 MFMAs, a barrier, a triangular one
// and one of 32, a barrier, where one workgroup per (head, chunk, 32 columns)
// and a launch a chunk took 31 us, each column block repeating the inverse. 2,048 positions of 32 heads:
// 1,020 -> 234 us (under a kernel trace, which adds to both, chunk_prep 67 and chunk_run 179: 5.6 a
// chunk); 100 positions of 4 heads 62.3 -> 34.4.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/lxm_chunk.h"
#include "lxm_math.h"

using namespace lxm;

namespace {

constexpr int CT = 256;  // threads per workgroup (4 waves: one per 16 positions)
constexpr int C = LXM_CHUNK;
constexpr int KL = 128;  // live key dims at most
constexpr int VD = 128;
constexpr int VT = 16;       // state columns per workgroup
constexpr int SK = KL + 4;   // row strides in floats: of rows read along k (16 rows on 16 bank groups),
constexpr int SR = KL + 16;  // of rows read across (4 rows x 16 columns on 64 banks),
constexpr int SC = C + 4;    // of the 64 x 64 matrices
constexpr int NTRI = 10;     // 16 x 16 tiles on or below the diagonal
// a (head, chunk)'s workspace in floats: W's 32 tiles and A2's 10 as A operands, U's 32 as D tiles,
// then eg, f and el
constexpr int WS_A2 = 32 * 256, WS_U = WS_A2 + NTRI * 256, WS_V = WS_U + 32 * 256;

typedef float v4f __attribute__((ext_vector_type(4)));

struct Vecs {
  float gc[C], beta[C], eg[C], f[C];  // (f = exp(g_last - gc))
  float el[4];                        // exp(g_last)
};
struct StepLds {  // B operands: the state's tiles and v_new
  v4f s[KL / 16][64], vn[4][64];
};
struct PrepLds {
  union {
    float kq[2][C][SK];  // k and q (blocks transposed), read by the Gram products; in their place
    struct {
      float kb[C][SR];   // k beta exp(gc), then v beta
      float lp[C][SC], tt[C][SC];
    };
  };
  v4f pt[4][64];         // per-wave scratch
  Vecs v;
};
struct RunLds {
  float k[C][SR], q[C][SK];
  StepLds st;
};
struct OneLds {
  float q[C][SK];
  union {
    float k[C][SK];
    float kb[C][SR];     // after the Gram products: k beta exp(gc), then k
  };
  union {
    float lp[C][SC];
    float w[C][SK];      // W (blocks transposed) once L is read
  };
  float tt[C][SC], a2[C][SC];
  v4f pt[4][64];
  Vecs v;
  StepLds st;
};
static_assert(2 * sizeof(PrepLds) <= 160 * 1024 && sizeof(OneLds) <= 160 * 1024, "LDS");
static_assert(LXM_CHUNK_WS == 4 * (WS_V + 2 * C + 4), "workspace");

__device__ __forceinline__ v4f mfma4(const v4f& a, const v4f& b, v4f c) {
#pragma unroll
  for (int r = 0; r < 4; r++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
  return c;
}
// A chain of MFMAs that ends inside a branch is waited for there: where the branch's end joined
// another path, the compiler has read the last MFMA's rows with no wait states in between (the last
// row of the tile came out without its last four terms).
__device__ __forceinline__ void settle(v4f& c) { asm volatile("s_nop 15" : "+v"(c)); }
__device__ __forceinline__ v4f ld4(const float* p) { return *reinterpret_cast<const v4f*>(p); }
__device__ __forceinline__ void st4(float* p, const v4f& v) { *reinterpret_cast<v4f*>(p) = v; }
__device__ __forceinline__ int wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
// what this wave's lanes stored in LDS, for its other lanes (a wave's LDS accesses run in order)
__device__ __forceinline__ void wave_sync() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_wave_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
__device__ __forceinline__ int tri(int ti, int tj) { return ti * (ti + 1) / 2 + tj; }
__device__ __forceinline__ void tri_of(int p, int& ti, int& tj) {
  ti = p < 1 ? 0 : p < 3 ? 1 : p < 6 ? 2 : 3;
  tj = p - ti * (ti + 1) / 2;
}
// column c of a row whose blocks of 16 are transposed as 4 x 4: lane group g's four k of a block
// are 16 consecutive bytes
__device__ __forceinline__ int pos16(int c) { return (c & ~15) | ((c & 3) << 2) | ((c >> 2) & 3); }
__device__ __forceinline__ void st_pos16(float* row, int d, const v4f& v) {  // d a multiple of 4
  float* p = row + (d & ~15) + ((d >> 2) & 3);
#pragma unroll
  for (int c = 0; c < 4; c++) p[4 * c] = v[c];
}
// element (i, j) of a tile as A operand: its float in the tile's 256
__device__ __forceinline__ int a_pos(int i, int j) {
  return ((i & 15) + 16 * (j & 3)) * 4 + ((j >> 2) & 3);
}
// a D tile as B operand into dst[64]
__device__ __forceinline__ void st_b(v4f* dst, const v4f& d) {
  const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
  float* p = reinterpret_cast<float*>(dst) + i16 * 4 + g;
#pragma unroll
  for (int r = 0; r < 4; r++) p[64 * r] = d[r];
}
// the block of 16 k from k0 of column c of rows of stride S, as B operand
template <int S>
__device__ __forceinline__ v4f ld_b(const float* m, int k0, int c) {
  const int g = (threadIdx.x & 63) >> 4;
  v4f b;
#pragma unroll
  for (int r = 0; r < 4; r++) b[r] = m[(k0 + 4 * r + g) * S + c];
  return b;
}
// the block of 16 k from k0 of row i of rows of stride SC, as A operand
__device__ __forceinline__ v4f ld_a(const float* m, int i, int k0) {
  const int g = (threadIdx.x & 63) >> 4;
  v4f a;
#pragma unroll
  for (int r = 0; r < 4; r++) a[r] = m[i * SC + k0 + 4 * r + g];
  return a;
}

// A chunk's n positions from p0, thread t: rows t / 32 + 8 j, dims 4 (t % 32) (below kl; rows past
// n: zero)
__device__ __forceinline__ void load_rows(const float* m, int64_t ts, int64_t off, int n,
                                          v4f (&x)[C / 8]) {
  const int d = 4 * (threadIdx.x & 31);
#pragma unroll
  for (int j = 0; j < C / 8; j++) {
    const int i = (threadIdx.x >> 5) + 8 * j, ic = i < n ? i : n - 1;
    x[j] = ld4(m + off + ic * ts + d);
  }
#pragma unroll
  for (int j = 0; j < C / 8; j++) {
    const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
    x[j] = (int)(threadIdx.x >> 5) + 8 * j < n ? x[j] : z;
  }
}
// rows (row(i), dims 4 (t % 32)) from x
template <class F>
__device__ __forceinline__ void each_row(F f) {
#pragma unroll
  for (int j = 0; j < C / 8; j++) f((int)(threadIdx.x >> 5) + 8 * j, 4 * (int)(threadIdx.x & 31), j);
}

// A2 and T of head h's chunk of n positions from p0, whose keys kv (load_rows) the caller holds. k,
// q: LDS rows of SK (blocks transposed); between() is called once they are read (by every wave) and
// before lp and tt are written; a2(i, j, x) stores A2[i][j] (tiles on or below the diagonal). After
// it every wave may read v, tt, and what between and a2 stored in LDS.
template <class FB, class FA>
__device__ __forceinline__ void prep(const lxm_chunk_io& io, int h, int64_t p0, int n,
                                     const v4f (&kv)[C / 8], float* k, float* q, float* lp,
                                     float* tt, v4f* pt, Vecs& v, FB between, FA a2) {
  const int t = threadIdx.x, w = wave(), lane = t & 63, i16 = lane & 15, g = lane >> 4;
  const int kl = io.kl;
  {
    v4f qv[C / 8];
    if (4 * (t & 31) < kl) {
      load_rows(io.q, io.qk_ts, p0 * io.qk_ts + (int64_t)(h / io.rl) * io.qk_hs, n, qv);
      each_row([&](int i, int d, int j) {
        st_pos16(k + i * SK, d, kv[j]);
        st_pos16(q + i * SK, d, qv[j]);
      });
    }
  }
  if (w == 0) {  // the vectors: position = lane. gc: binary64 sums in order, each prefix rounded
    float b = 0.0f, gr = 0.0f;
    if (lane < n) {
      b = io.beta[(p0 + lane) * io.g_ts + (int64_t)h * io.g_hs];
      gr = io.g[(p0 + lane) * io.gl_ts + h];
    }
    double a = 0.0;
    float gc = 0.0f;
#pragma unroll
    for (int i = 0; i < C; i++) {
      a += (double)__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(gr), i));
      gc = lane == i ? (float)a : gc;
    }
    const float gl = (float)a;
    v.gc[lane] = gc;
    v.beta[lane] = b;
    v.eg[lane] = cr_exp(gc);
    v.f[lane] = cr_exp(gl - gc);
    if (lane == 0) v.el[0] = cr_exp(gl);
  }
  lds_barrier();
  // ---- the Gram tiles, dealt to the waves
  v4f aq[3], ak[3];
#pragma unroll
  for (int u = 0; u < 3; u++) {
    aq[u] = ak[u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const int p = w + 4 * u;
    if (p >= NTRI) continue;
    int ti, tj;
    tri_of(p, ti, tj);
    const float bi = v.beta[16 * ti + i16];
    const float *qi = q + (16 * ti + i16) * SK + 4 * g, *ki = k + (16 * ti + i16) * SK + 4 * g,
                *kj = k + (16 * tj + i16) * SK + 4 * g;
    v4f a = ld4(qi), b = ld4(ki), c = ld4(kj);
    for (int d0 = 0; d0 < kl; d0 += 16) {
      const int dn = d0 + 16 < kl ? d0 + 16 : d0;  // (the last block again, unused)
      const v4f an = ld4(qi + dn), bn = ld4(ki + dn), cn = ld4(kj + dn);
      aq[u] = mfma4(a, c, aq[u]);
      ak[u] = mfma4(b * bi, c, ak[u]);
      a = an;
      b = bn;
      c = cn;
    }
    settle(aq[u]);
    settle(ak[u]);
  }
  lds_barrier();
  between();
#pragma unroll
  for (int u = 0; u < 3; u++) {
    const int p = w + 4 * u;
    if (p >= NTRI) continue;
    int ti, tj;
    tri_of(p, ti, tj);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = 16 * ti + 4 * g + r, j = 16 * tj + i16;
      const float gm = j <= i ? cr_exp(v.gc[i] - v.gc[j]) : 0.0f;
      a2(i, j, aq[u][r] * gm);
      lp[i * SC + j] = j < i ? ak[u][r] * gm : 0.0f;
    }
  }
  lds_barrier();
  // ---- T: diagonal block w by forward substitution, lane % 16 its column in registers
  {
    const float* lb = lp + 16 * w * SC + 16 * w;
    float tc[16];
    tc[0] = i16 == 0 ? 1.0f : 0.0f;
#pragma unroll
    for (int i = 1; i < 16; i++) {
      float s = 0.0f;
#pragma unroll
      for (int m4 = 0; m4 < (i + 3) / 4; m4++) {
        const v4f l4 = ld4(lb + i * SC + 4 * m4);
#pragma unroll
        for (int m = 0; m < 4; m++)
          if (4 * m4 + m < i) s = s + l4[m] * tc[4 * m4 + m];
      }
      tc[i] = i16 < i ? -s : i16 == i ? 1.0f : 0.0f;
    }
    if (lane < 16) {
#pragma unroll
      for (int i = 0; i < 16; i++) tt[(16 * w + i) * SC + 16 * w + i16] = tc[i];
    }
  }
  lds_barrier();
  // block rows 1..3: T_ij = -T_ii P, P = sum_{m=j}^{i-1} L_im T_mj; block (i, j) on wave j
  for (int bi = 1; bi < 4; bi++) {
    if (w < bi) {
      const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
      v4f p = z;
      for (int m = w; m < bi; m++)
        p = mfma4(ld_a(lp, 16 * bi + i16, 16 * m), ld_b<SC>(tt, 16 * m, 16 * w + i16), p);
      settle(p);
      st_b(pt + 64 * w, p);
      wave_sync();
      v4f x = mfma4(ld_a(tt, 16 * bi + i16, 16 * bi), pt[64 * w + lane], z);
      settle(x);
#pragma unroll
      for (int r = 0; r < 4; r++) tt[(16 * bi + 4 * g + r) * SC + 16 * w + i16] = -x[r];
    }
    lds_barrier();
  }
}
// tile (ti, column block at c) of T times rows of stride SR (T is lower triangular: k blocks <= ti)
__device__ __forceinline__ v4f t_times(const float* tt, const float* m, int ti, int c) {
  const int i16 = threadIdx.x & 15;
  v4f a = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int kb = 0; kb < 4; kb++)
    if (kb <= ti) a = mfma4(ld_a(tt, 16 * ti + i16, 16 * kb), ld_b<SR>(m, 16 * kb, c + i16), a);
  return a;
}

// One chunk's step for 16 state columns: wave w holds positions 16 w .. 16 w + 15 and state tiles
// 2 w and 2 w + 1 (s; every tile in st.s as B operand). wa, qa, aa(t): the wave's rows of W, q
// exp(gc) and A2 as A operands; u: U's tile; k: the chunk's keys, rows of SR in LDS; f[t][r] of
// position 16 t + 4 r + g. mid(): after W, q and U are read. Returns o's tile; the new state in s and
// st.s (behind a barrier of the caller's).
template <class WA, class QA, class AA, class Mid>
__device__ __forceinline__ v4f chunk_step(StepLds& st, const float* k, int nkt, WA wa, QA qa,
                                          const v4f& u, const v4f (&f)[4], float el, AA aa,
                                          v4f (&s)[2], Mid mid) {
  const int w = wave(), lane = threadIdx.x & 63, i16 = lane & 15;
  const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
  v4f vp = z, o1 = z;
#pragma unroll
  for (int t = 0; t < KL / 16; t++) {  // (zeros past kl)
    const v4f b = st.s[t][lane];
    vp = mfma4(wa(t), b, vp);
    o1 = mfma4(qa(t), b, o1);
  }
  st_b(st.vn[w], u - vp);
  mid();
  lds_barrier();
  v4f b[4], x[2] = {z, z};
#pragma unroll
  for (int t = 0; t < 4; t++) b[t] = st.vn[t][lane];
  v4f a = mfma4(aa(0), b[0], z);
  if (w > 0) {
    a = mfma4(aa(1), b[1], a);
    if (w > 1) {
      a = mfma4(aa(2), b[2], a);
      if (w > 2) a = mfma4(aa(3), b[3], a);
      settle(a);
    }
    settle(a);
  }
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int j = 0; j < 2; j++)
      x[j] = mfma4(ld_b<SR>(k, 16 * t, 16 * (2 * w + j) + i16) * f[t], b[t], x[j]);
#pragma unroll
  for (int j = 0; j < 2; j++) {
    x[j] = s[j] * el + x[j];
    s[j] = 2 * w + j < nkt ? x[j] : z;
    st_b(st.s[2 * w + j], s[j]);
  }
  return o1 + a;
}

__device__ __forceinline__ float* state_of(const lxm_chunk_io& io, int h, int c0) {
  return io.S + ((size_t)(h / io.rl) * io.rfull + h % io.rl) * 256 * VD + c0;
}
// (STAGE: each tile into st.s as it comes)
template <bool STAGE>
__device__ __forceinline__ void load_state(const float* S, int nkt, StepLds& st, v4f (&s)[2]) {
  const int w = wave(), lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    s[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    if (2 * w + j < nkt) {
#pragma unroll
      for (int r = 0; r < 4; r++) s[j][r] = S[(size_t)(16 * (2 * w + j) + 4 * g + r) * VD + i16];
    }
    if constexpr (STAGE) st_b(st.s[2 * w + j], s[j]);
  }
}
__device__ __forceinline__ void store_state(float* S, int nkt, const v4f (&s)[2]) {
  const int w = wave(), lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int j = 0; j < 2; j++)
    if (2 * w + j < nkt) {
#pragma unroll
      for (int r = 0; r < 4; r++) S[(size_t)(16 * (2 * w + j) + 4 * g + r) * VD + i16] = s[j][r];
    }
}
__device__ __forceinline__ void store_o(const lxm_chunk_io& io, int h, int c0, int64_t p0, int n,
                                        const v4f& o) {
  const int w = wave(), lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int i = 16 * w + 4 * g + r;
    if (i < n)
      io.o[(p0 + i) * io.o_ts + (int64_t)h * VD + c0 + i16] = io.o_bf16 ? bf16r(o[r]) : o[r];
  }
}
// (workgroups are dealt to the 8 XCDs in turn: a head's column groups, NB blocks of VT columns each, on
// one of them, whose L2 then holds its keys, queries, T and A2)
template <int NB>
__device__ __forceinline__ bool head_cols(int n_slots, int& h, int& c0) {
  constexpr int G = VD / (VT * NB);
  const int x = blockIdx.x & 7, j = blockIdx.x >> 3;
  h = x + 8 * (j / G);
  c0 = (j % G) * VT * NB;
  return h < n_slots;
}

}  // namespace

// W, U, A2 and the vectors of every (head, chunk), chunks ch0 .. ch0 + gridDim.y - 1 of T positions
__global__ __launch_bounds__(CT, 2) void chunk_prep(lxm_chunk_io io, int T, int ch0, float* ws) {
  extern __shared__ __align__(16) uint8_t smem_raw[];
  PrepLds& l = *reinterpret_cast<PrepLds*>(smem_raw);
  const int h = blockIdx.x, ch = ch0 + blockIdx.y, n = T - ch * C < C ? T - ch * C : C;
  const int w = wave(), lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
  const int64_t p0 = (int64_t)ch * C;
  const bool mine = 4 * (int)(threadIdx.x & 31) < io.kl;
  float* o = ws + ((size_t)blockIdx.y * io.n_slots + h) * (LXM_CHUNK_WS / 4);
  v4f kv[C / 8], vv[C / 8];
  if (mine) load_rows(io.k, io.qk_ts, p0 * io.qk_ts + (int64_t)(h / io.rl) * io.qk_hs, n, kv);
  prep(io, h, p0, n, kv, &l.kq[0][0][0], &l.kq[1][0][0], &l.lp[0][0], &l.tt[0][0], &l.pt[0][0], l.v,
       [&] {
         if (mine)
           each_row([&](int i, int d, int j) {
             st4(&l.kb[i][d], (kv[j] * l.v.beta[i]) * l.v.eg[i]);
           });
         load_rows(io.v, io.v_ts, p0 * io.v_ts + (int64_t)h * VD, n, vv);
       },
       [&](int i, int j, float x) { o[WS_A2 + tri(i >> 4, j >> 4) * 256 + a_pos(i, j)] = x; });
  // wave w: the column blocks w and w + 4 of W, then of U
  for (int tc = w; 16 * tc < io.kl; tc += 4)
#pragma unroll
    for (int ti = 0; ti < 4; ti++) {
      const v4f a = t_times(&l.tt[0][0], &l.kb[0][0], ti, 16 * tc);
#pragma unroll
      for (int r = 0; r < 4; r++) o[(ti * 8 + tc) * 256 + a_pos(4 * g + r, i16)] = a[r];
    }
  lds_barrier();  // (kb is read)
  each_row([&](int i, int d, int j) { st4(&l.kb[i][d], vv[j] * l.v.beta[i]); });
  lds_barrier();
  for (int tc = w; tc < VD / 16; tc += 4)
#pragma unroll
    for (int ti = 0; ti < 4; ti++)
      st4(o + WS_U + (ti * 8 + tc) * 256 + 4 * lane, t_times(&l.tt[0][0], &l.kb[0][0], ti, 16 * tc));
  if (threadIdx.x < C) {
    o[WS_V + threadIdx.x] = l.v.eg[threadIdx.x];
    o[WS_V + C + threadIdx.x] = l.v.f[threadIdx.x];
    if (threadIdx.x == 0) o[WS_V + 2 * C] = l.v.el[0];
  }
}

// the chunks ch0 .. ch0 + nch - 1 in order for 16 state columns of a head; each operand is
// requested for the next chunk right after its last use
__global__ __launch_bounds__(CT, 1) void chunk_run(lxm_chunk_io io, int T, int ch0, int nch,
                                                   const float* ws) {
  __shared__ RunLds l;
  int h, c0;
  if (!head_cols<1>(io.n_slots, h, c0)) return;
  const int w = wave(), lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
  const int nkt = io.kl / 16, kh = h / io.rl, row = 16 * w + i16;
  float* S = state_of(io, h, c0);
  v4f s[2], wa[KL / 16], ka[KL / 16], qa[KL / 16], ar[4], f[4], u;
  float eg, el;
  auto wsc = [&](int c) { return ws + ((size_t)c * io.n_slots + h) * (LXM_CHUNK_WS / 4); };
  auto get_kq = [&](int c) {  // (positions past the end: the last, taken as zero below)
    const int p = (ch0 + c) * C + row;
    const int64_t o = (int64_t)(p < T ? p : T - 1) * io.qk_ts + (int64_t)kh * io.qk_hs + 4 * g;
    const float* x = wsc(c);
#pragma unroll
    for (int t = 0; t < KL / 16; t++) {  // (blocks past kl: the last one's, taken as zero)
      const int tk = t < nkt ? t : nkt - 1;
      ka[t] = ld4(io.k + o + 16 * tk);
      qa[t] = ld4(io.q + o + 16 * tk);
      wa[t] = ld4(x + (w * 8 + tk) * 256 + 4 * lane);
    }
    eg = x[WS_V + row];
    u = ld4(x + WS_U + (w * 8 + c0 / 16) * 256 + 4 * lane);
  };
  auto get_rest = [&](int c) {
    const float* x = wsc(c);
#pragma unroll
    for (int t = 0; t < 4; t++) {
      if (t <= w) ar[t] = ld4(x + WS_A2 + tri(w, t) * 256 + 4 * lane);
#pragma unroll
      for (int r = 0; r < 4; r++) f[t][r] = x[WS_V + C + 16 * t + 4 * r + g];
    }
    el = x[WS_V + 2 * C];
  };
  load_state<true>(S, nkt, l.st, s);
  get_kq(0);
  get_rest(0);
  lds_barrier();
  for (int c = 0; c < nch; c++) {
    const int p0 = (ch0 + c) * C, n = T - p0 < C ? T - p0 : C;
    const int cn = c + 1 < nch ? c + 1 : c;  // (the last chunk's again, unused)
    const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < KL / 16; t++) {
      const bool in = row < n && t < nkt;
      st4(&l.k[row][16 * t + 4 * g], in ? ka[t] : z);
      st_pos16(l.q[row], 16 * t + 4 * g, in ? qa[t] * eg : z);
      wa[t] = t < nkt ? wa[t] : z;
    }
    wave_sync();  // (a wave reads its own rows of q)
    const v4f o = chunk_step(
        l.st, &l.k[0][0], nkt, [&](int t) { return wa[t]; },
        [&](int t) { return ld4(&l.q[row][16 * t + 4 * g]); }, u, f, el,
        [&](int t) { return ar[t]; }, s, [&] { get_kq(cn); });
    store_o(io, h, c0, p0, n, o);
    get_rest(cn);
    lds_barrier();  // (the state's tiles for every wave; k and v_new are read)
  }
  store_state(S, nkt, s);
}

// one chunk of every head: A2, T and W repeated by each of a head's VD / (VT NB) workgroups, each with
// its own columns of U and its NB steps one after the other (one block's tiles in LDS at a time)
template <int NB>
__global__ __launch_bounds__(CT, 1) void chunk_one(lxm_chunk_io io) {
  extern __shared__ __align__(16) uint8_t smem_raw[];
  OneLds& l = *reinterpret_cast<OneLds*>(smem_raw);
  int h, c0;
  if (!head_cols<NB>(io.n_slots, h, c0)) return;
  const int w = wave(), lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
  const int nkt = io.kl / 16, n = io.n, row = 16 * w + i16;
  const bool mine = 4 * (int)(threadIdx.x & 31) < io.kl;
  float* S = state_of(io, h, c0);
  v4f kv[C / 8], s[NB][2], vb[NB][4], f[4];
  if (mine) {
    load_rows(io.k, io.qk_ts, (int64_t)(h / io.rl) * io.qk_hs, n, kv);
  } else {  // (dims past kl: zero in every product)
    const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
    each_row([&](int i, int d, int j) {
      kv[j] = z;
      st4(&l.q[i][d], z);
    });
  }
#pragma unroll
  for (int cb = 0; cb < NB; cb++) {
#pragma unroll
    for (int t = 0; t < 4; t++)  // v's 16 columns as B operand
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = 16 * t + 4 * r + g;
        vb[cb][t][r] = i < n ? io.v[i * io.v_ts + (int64_t)h * VD + c0 + VT * cb + i16] : 0.0f;
      }
    if (cb == 0) load_state<true>(S, nkt, l.st, s[0]);
    else load_state<false>(S + VT * cb, nkt, l.st, s[cb]);
  }
  prep(io, h, 0, n, kv, &l.k[0][0], &l.q[0][0], &l.lp[0][0], &l.tt[0][0], &l.pt[0][0], l.v,
       [&] {
         each_row([&](int i, int d, int j) {
           st4(&l.kb[i][d], (kv[j] * l.v.beta[i]) * l.v.eg[i]);
         });
       },
       [&](int i, int j, float x) { l.a2[i][j] = x; });
#pragma unroll 1
  for (int tc = w; tc < KL / 16; tc += 4)
#pragma unroll
    for (int ti = 0; ti < 4; ti++) {
      const v4f a = t_times(&l.tt[0][0], &l.kb[0][0], ti, 16 * tc);
#pragma unroll
      for (int r = 0; r < 4; r++) l.w[16 * ti + 4 * g + r][pos16(16 * tc + i16)] = a[r];
    }
  v4f u[NB];
#pragma unroll
  for (int cb = 0; cb < NB; cb++) u[cb] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int t = 0; t < 4; t++) {
    v4f b[NB];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = 16 * t + 4 * r + g;
#pragma unroll
      for (int cb = 0; cb < NB; cb++) b[cb][r] = vb[cb][t][r] * l.v.beta[i];
      f[t][r] = l.v.f[i];
    }
    if (t <= w) {
      const v4f a = ld_a(&l.tt[0][0], row, 16 * t);
#pragma unroll
      for (int cb = 0; cb < NB; cb++) {
        u[cb] = mfma4(a, b[cb], u[cb]);
        settle(u[cb]);
      }
    }
  }
  lds_barrier();  // (kb is read: the keys in its place, behind the step's barrier)
  each_row([&](int i, int d, int j) { st4(&l.kb[i][d], kv[j]); });
  const float eg = l.v.eg[row];
#pragma unroll
  for (int cb = 0; cb < NB; cb++) {
    if (cb > 0) {  // (the block before has read its state before its step's barrier, v_new by this one)
#pragma unroll
      for (int j = 0; j < 2; j++) st_b(l.st.s[2 * w + j], s[cb][j]);
      lds_barrier();
    }
    const v4f o = chunk_step(
        l.st, &l.kb[0][0], nkt, [&](int t) { return ld4(&l.w[row][16 * t + 4 * g]); },
        [&](int t) { return ld4(&l.q[row][16 * t + 4 * g]) * eg; }, u[cb], f, l.v.el[0],
        [&](int t) { return ld_a(&l.a2[0][0], row, 16 * t); }, s[cb], [] {});
    store_o(io, h, c0 + VT * cb, 0, n, o);
    store_state(S + VT * cb, nkt, s[cb]);
  }
}

// q, k, v and S are read four floats at a time: their pointers 16-byte aligned, and the strides
// between those reads multiples of 4 floats
static bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }
static bool io_ok(const lxm_chunk_io* io) {
  return io && io->kl >= 1 && io->kl <= KL && io->kl % 16 == 0 && io->n_slots >= 1 && io->rl >= 1 &&
         io->rfull >= io->rl && al16(io->q) && al16(io->k) && al16(io->v) && al16(io->S) &&
         io->qk_ts % 4 == 0 && io->qk_hs % 4 == 0 && io->v_ts % 4 == 0;
}
static int cols_grid(int n_slots, int nb) { return (n_slots + 7) / 8 * 8 * (VD / (VT * nb)); }

template <int NB>
static int launch_one(const lxm_chunk_io* io, hipStream_t st) {
  const int lds = (int)sizeof(OneLds);
  const hipError_t e = hipFuncSetAttribute((const void*)chunk_one<NB>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(chunk_one<NB>, dim3(cols_grid(io->n_slots, NB)), dim3(CT), lds, st, *io);
  return (int)hipGetLastError();
}

extern "C" int lxm_gdn_chunk(const lxm_chunk_io* io, void* stream) {
  if (!io_ok(io) || io->n < 1 || io->n > C) return (int)hipErrorInvalidValue;
  // OneLds fills a CU, so a workgroup past the 256th waits for a whole one's time: up to 32 heads 16
  // columns a workgroup (64 positions of 32 heads 25.1 us), from there on 32, half as many workgroups,
  // each a step longer (34 heads 29.3 us, 47.2 in 16 columns; 64 heads 29.6 and 48.2; 128 heads 57.1
  // and 94.4)
  const bool wide = io->n_slots > 256 / (VD / VT);
  return wide ? launch_one<2>(io, (hipStream_t)stream) : launch_one<1>(io, (hipStream_t)stream);
}

extern "C" int lxm_gdn_chunks(const lxm_chunk_io* io, int T, void* ws, int64_t ws_bytes,
                              void* stream) {
  if (!io_ok(io) || T < 1 || !al16(ws)) return (int)hipErrorInvalidValue;
  const int64_t per = (int64_t)LXM_CHUNK_WS * io->n_slots;
  const int nch = (int)(((int64_t)T + C - 1) / C);
  int64_t grp = ws ? ws_bytes / per : 0;  // chunks the workspace holds
  if (grp < 1) return (int)hipErrorInvalidValue;
  if (grp > 65535) grp = 65535;  // (a grid's y extent)
  const int lds = (int)sizeof(PrepLds);
  const hipError_t e = hipFuncSetAttribute((const void*)chunk_prep,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return (int)e;
  for (int c = 0; c < nch; c += (int)grp) {
    const int m = nch - c < grp ? nch - c : (int)grp;
    hipLaunchKernelGGL(chunk_prep, dim3(io->n_slots, m), dim3(CT), lds, (hipStream_t)stream, *io, T, c,
                       static_cast<float*>(ws));
    hipLaunchKernelGGL(chunk_run, dim3(cols_grid(io->n_slots, 1)), dim3(CT), 0, (hipStream_t)stream,
                       *io, T, c, m, static_cast<const float*>(ws));
  }
  return (int)hipGetLastError();
}
