// Bit-exact KV data movement on gfx950: paged append (scatter into slots), paged
// gather (pages -> contiguous rows) and the index gather/scatter of a contiguous
// [B, H, S, D] cache.  Elements are moved as raw 16/32-bit words, so every
// kernel here is exact for any dtype of that size.
//
// All kernels are HBM-bound copies: each thread moves one 16-byte chunk
// (8 half / 4 float elements) per row, so a wavefront reads or writes 1 KiB
// per instruction in the layout-favoured direction.
#include "ivakv_internal.h"

namespace ivakv {
namespace {

struct alignas(16) Chunk16 {
  uint32_t w[4];
};

// ---------------------------------------------------------------------------
// append: new rows [n_tok][Hkv][D] (strided) -> k_pool / v_pool slots
// ---------------------------------------------------------------------------
struct AppendArgs {
  const void* k_new;
  const void* v_new;
  int64_t kts, khs, vts, vhs;  // element strides (token, head)
  void* k_pool;
  void* v_pool;
  const int32_t* slots;
  int n_tok, Hkv, D, bs;
  int64_t n_slots;  // num_pages * bs
};

// Element path (sources or pools not 16-byte aligned): one thread per (token, head,
// chunk of X elements).  Thread order (token % 16, chunk, head, token / 16): the 16
// lanes of a token group cover 16 consecutive tokens, which a chunk append puts in
// consecutive slots of one page, so their K elements are 256 contiguous bytes per
// chunk and each V dim's elements one 32-byte row.
template <typename E>
__global__ __launch_bounds__(256) void append_kernel(AppendArgs a) {
  constexpr int X = 16 / sizeof(E);
  const int nch = a.D / X;
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = (int64_t)cdiv(a.n_tok, 16) * 16 * a.Hkv * nch;
  if (gid >= total) return;
  const int t_lo = (int)(gid & 15);
  const int64_t g1 = gid >> 4;
  const int c = (int)(g1 % nch);
  const int64_t g2 = g1 / nch;
  const int h = (int)(g2 % a.Hkv);
  const int64_t t = (g2 / a.Hkv) * 16 + t_lo;
  if (t >= a.n_tok) return;
  const int64_t slot = a.slots[t];
  if (slot < 0 || slot >= a.n_slots) return;
  const int64_t page = slot / a.bs;
  const int off = (int)(slot - page * a.bs);
  const int64_t head_base = page * a.Hkv + h;
  const E* ks = static_cast<const E*>(a.k_new) + t * a.kts + h * a.khs + (int64_t)c * X;
  const E* vs = static_cast<const E*>(a.v_new) + t * a.vts + h * a.vhs + (int64_t)c * X;
  E* kd = static_cast<E*>(a.k_pool) + ((head_base * nch + c) * a.bs + off) * X;
  E* vd = static_cast<E*>(a.v_pool) + head_base * a.D * a.bs + (int64_t)c * X * a.bs + off;
#pragma unroll
  for (int i = 0; i < X; ++i) kd[i] = ks[i];
#pragma unroll
  for (int i = 0; i < X; ++i) vd[(int64_t)i * a.bs] = vs[i];
}

// 16-byte path: one thread per (token, group of up to kAppendHeads kv heads, 16-byte
// chunk), thread order (token % 16, chunk, head group, token / 16).  A lane issues the
// K and V loads of all its heads before the first store, so a wave keeps 16 KiB of
// source rows in flight and a chunk append runs in about one round of resident waves
// (one head per lane: eight rounds of single round trips).  K chunks are stored whole
// (256 contiguous bytes per 16 consecutive slots); each V chunk is spread over X rows
// of the page's [D][bs] tile.  Row loads and K stores carry the non-temporal hint
// (8192 rows from HBM: 14.9 µs against 17.7 µs with neither).  Blocks run in
// XCD-contiguous order (xcd_contiguous_block).  Groups of 32 or 64 consecutive tokens
// per lane group (fewer split pages, 16 / 32 bytes per token per load) measured
// 21 / 33 µs against 14.8 µs on 8192 aligned rows.
// Few rows (a decode step's one token per sequence, each to its own page; short
// chunks): one head per lane in 64-thread workgroups (HEADS = 1), so the stores spread
// over many CUs instead of the few workgroups eight heads per lane would give.  Rows of
// 8 kv heads x 128 dims from HBM: a 32-sequence decode step 14.0 -> 2.9 us, 256
// sequences 16.4 -> 5.7 us, one 512-row chunk 6.1 -> 3.2 us, 2048 rows 7.6 -> 7.1 us;
// at 8192 rows eight heads per lane stay ahead (15.6 against 18.5 us).
constexpr int kAppendHeads = 8;
constexpr int64_t kFewAppendThreads = 1024 * 64;  // below 1024 waves: one head per lane

template <typename E, int HEADS>
__global__ __launch_bounds__(256) void append_vec_kernel(AppendArgs a) {
  constexpr int X = 16 / sizeof(E);
  const int nch = a.D / X;
  const int ngrp = cdiv(a.Hkv, HEADS);
  const int64_t gid = xcd_contiguous_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (gid >= (int64_t)cdiv(a.n_tok, 16) * 16 * ngrp * nch) return;
  const int t_lo = (int)(gid & 15);
  const int64_t g1 = gid >> 4;
  const int c = (int)(g1 % nch);
  const int64_t g2 = g1 / nch;
  const int h0 = (int)(g2 % ngrp) * HEADS;
  const int64_t t = (g2 / ngrp) * 16 + t_lo;
  if (t >= a.n_tok) return;
  const int64_t slot = a.slots[t];
  if (slot < 0 || slot >= a.n_slots) return;
  const int64_t page = slot / a.bs;
  const int off = (int)(slot - page * a.bs);
  const int nh = min(HEADS, a.Hkv - h0);
  const E* ks = static_cast<const E*>(a.k_new) + t * a.kts + (int64_t)c * X;
  const E* vs = static_cast<const E*>(a.v_new) + t * a.vts + (int64_t)c * X;
  union Row {
    Chunk16 c16;
    E e[X];
  };
  Row k[HEADS], v[HEADS];
#pragma unroll
  for (int u = 0; u < HEADS; ++u) {
    if (u < nh) {
      k[u].c16 = ld<true, Chunk16>(ks + (h0 + u) * a.khs);
      v[u].c16 = ld<true, Chunk16>(vs + (h0 + u) * a.vhs);
    }
  }
#pragma unroll
  for (int u = 0; u < HEADS; ++u) {
    if (u < nh) {
      const int64_t head_base = page * a.Hkv + h0 + u;
      E* kd = static_cast<E*>(a.k_pool) + ((head_base * nch + c) * a.bs + off) * X;
      E* vd = static_cast<E*>(a.v_pool) + head_base * a.D * a.bs + (int64_t)c * X * a.bs + off;
      st<true, Chunk16>(kd, k[u].c16);
#pragma unroll
      for (int i = 0; i < X; ++i) vd[(int64_t)i * a.bs] = v[u].e[i];
    }
  }
}

// Whole pages of 16-bit rows (16-row pages, head_dim 64 / 128 / 256, 16-byte rows): a wave
// takes one kv head of 16 tokens that fill one page, so that its V page is written as 16-byte
// chunks.  What bounds append_vec_kernel on a chunk append is the number of its V stores,
// eight 2-byte stores per lane and chunk, each of four 32-byte runs; here V's rows pass through
// LDS and come back transposed (ds_read_b64_tr_b16: lane i of 16 gets column i of four rows).
//
// Which tokens fill a page is found per window of 16 tokens, from the slots of the windows
// around it: a run starts at a token whose slot opens a page and whose 15 successors have the
// next slots.  Runs never overlap, so at most one starts in a window and belongs to it
// (running into the next); tokens of no run (a chunk's ends, decode tokens, scattered or
// repeated slots) are stored element by element by their own window.  Every row load of a wave
// is issued before its first store; windows x kv heads go in XCD-contiguous order, one head
// per wave (two: 15.0 against 12.0 us on the ragged chunks below).
//
// us against append_vec_kernel, 8 heads x 128 dims from HBM: 11 ragged chunks (4658 rows) 12.0 :
// 16.7, 8 chunks of 4096 53.7 : 64.9, 16 of 512 15.1 : 15.1, starting mid-page 17.5 : 19.0, 300
// of 20 18.6 : 22.2; 32 heads, 16 chunks of 512 mid-page 52 : 84; 16 heads x 64, 16 of 512 14.3 :
// 15.6.  Chosen from kRunTokens rows and kRunElems elements of K up: below, a window's one wave
// per head is a long chain (512 rows of 8 heads 4.7 : 3.4, 2048 6.3 : 7.6; a decode step of 1024
// scattered rows 13.2 : 11.0); head_dim 256 from four times that (300 x 20 rows 21.3 : 20.4, 16
// chunks of 512 13.6 : 17.7).  Rows scattered singly gain little (8192 of them 69.6 : 70.2, of
// 32 heads 304 : 317; 2048 of 8 heads 19.0 : 20.7, of 32 heads 71.3 : 70.5).
typedef short i16x4_t __attribute__((ext_vector_type(4)));
constexpr int kRunTokens = 2048;
constexpr int64_t kRunElems = 1 << 21;

template <int D>
__global__ __launch_bounds__(256) void append_runs_kernel(AppendArgs a) {
  constexpr int NCH = D / 8;       // 16-byte chunks of a row
  constexpr int NL = NCH / 4;      // loads per lane of 16 rows
  constexpr int kRow = D + 16;     // LDS row in elements (32 bytes of padding spread the rows)
  __shared__ __attribute__((aligned(16))) uint16_t s_v[4][16 * kRow];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int groups = cdiv(a.Hkv, 4);
  const int64_t blk = xcd_contiguous_block(blockIdx.x, gridDim.x);
  const int64_t g = blk / groups;
  const int h = (int)(blk - g * groups) * 4 + wave;
  if (h >= a.Hkv) return;

  // Slots of tokens 16 g - 16 .. 16 g + 47, one per lane; the window is lanes 16 .. 31.
  const int64_t tl = 16 * g - 16 + lane;
  const int64_t slot = tl >= 0 && tl < a.n_tok ? (int64_t)a.slots[tl] : -1;
  const bool valid = slot >= 0 && slot < a.n_slots;
  const int next = __shfl_down((int)slot, 1);
  uint64_t run = __ballot(valid && lane < 63 && next == (int)slot + 1);
  run &= run >> 1;
  run &= run >> 2;
  run &= run >> 4;
  run &= run >> 7;  // lanes whose next 15 tokens have the next 15 slots
  const uint64_t starts = run & __ballot(valid && (slot & 15) == 0);
  const uint64_t own = starts & 0xFFFF0000u, before = starts & 0xFFFFu;
  uint64_t left = __ballot(valid) & 0xFFFF0000u;
  if (before) left &= ~(0xFFFFull << __builtin_ctzll(before));
  if (own) left &= ~(0xFFFFull << __builtin_ctzll(own));

  const uint16_t* kn = static_cast<const uint16_t*>(a.k_new) + h * a.khs;
  const uint16_t* vn = static_cast<const uint16_t*>(a.v_new) + h * a.vhs;
  uint16_t* kp = static_cast<uint16_t*>(a.k_pool);
  uint16_t* vp = static_cast<uint16_t*>(a.v_pool);
  // The leftover tokens of this window: token lane % 16, chunks 4 i + lane / 16.
  const int t_lo = lane & 15, c_lo = lane >> 4;
  const int64_t s_left = __shfl((int)slot, 16 + t_lo);
  const bool is_left = ((left >> (16 + t_lo)) & 1) != 0;
  union Row {
    Chunk16 c16;
    uint16_t e[8];
  };
  Row lk[NL], lv[NL];
  auto load_left = [&]() {
    const int64_t t = 16 * g + t_lo;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      lk[i].c16 = load_nt<Chunk16>(kn + t * a.kts + 8 * (4 * i + c_lo));
      lv[i].c16 = load_nt<Chunk16>(vn + t * a.vts + 8 * (4 * i + c_lo));
    }
  };
  if (own) {
    const int l0 = __builtin_ctzll(own);
    const int64_t t0 = 16 * g - 16 + l0;
    const int64_t page = (int64_t)__shfl((int)slot, l0) >> 4;
    Chunk16 k[NL], v[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      // K: lanes along the tokens of a chunk, as its page lies; V: along a token's row.
      k[i] = load_nt<Chunk16>(kn + (t0 + t_lo) * a.kts + 8 * (4 * i + c_lo));
      v[i] = load_nt<Chunk16>(vn + (t0 + (64 * i + lane) / NCH) * a.vts + 8 * ((64 * i + lane) % NCH));
    }
    if (is_left) load_left();
    const int64_t tile = (page * a.Hkv + h) * (16 * D);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      *reinterpret_cast<Chunk16*>(&s_v[wave][(64 * i + lane) / NCH * kRow + 8 * ((64 * i + lane) % NCH)]) = v[i];
      store_nt(kp + tile + 8 * (64 * i + lane), k[i]);
    }
    __builtin_amdgcn_wave_barrier();  // (a wave's LDS accesses take effect in order)
    // Chunk (dim, half): the 8 tokens 8 half .. of a dim, from two transposed reads of
    // four rows by 16 dims.
    const int half = c_lo & 1;
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
      typedef __attribute__((address_space(3))) i16x4_t lds_i16x4;
      const int d0 = 32 * i + 16 * (lane >> 5);
      const uint16_t* src = &s_v[wave][(8 * half + (t_lo >> 2)) * kRow + d0 + 4 * (t_lo & 3)];
      const uint64_t lo = __builtin_bit_cast(uint64_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)src));
      const uint64_t hi =
          __builtin_bit_cast(uint64_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(src + 4 * kRow)));
      const Chunk16 o{{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)}};
      store_nt(vp + tile + (d0 + t_lo) * 16 + 8 * half, o);
    }
  } else if (is_left) {
    load_left();
  }
  if (is_left) {
    const int row = (int)s_left & 15;
    const int64_t tile = ((s_left >> 4) * a.Hkv + h) * (16 * D);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int c = 4 * i + c_lo;
      store_nt(kp + tile + (16 * c + row) * 8, lk[i].c16);
#pragma unroll
      for (int e = 0; e < 8; ++e) vp[tile + (8 * c + e) * 16 + row] = lv[i].e[e];
    }
  }
}

// ---------------------------------------------------------------------------
// gather: pages -> k_out / v_out = [B][Hkv][out_len][D]
// ---------------------------------------------------------------------------
struct GatherArgs {
  const void* k_pool;
  const void* v_pool;
  const int32_t* bt;
  const int32_t* ctx;
  int max_blocks, Hkv, D, bs, num_pages, out_len;
  void* k_out;
  void* v_out;
};

// Any element size, page size and head_dim (gather16_kernel takes 2-byte elements on
// 16-row pages at head_dim 64 / 128 / 256).  Grid (logical page, group of H kv heads,
// sequence), 256 threads per kv head.  Thread index (within a head) = chunk * bs + row, so
// the K page (stored [D/X][bs][X]) is read as one contiguous run and each
// 16-byte V chunk is assembled from X row-adjacent elements of the [D][bs]
// page (consecutive lanes read consecutive rows).  K reads carry the non-temporal hint
// (each page is read once); the output stores do not (C2 batch at one kv head per
// workgroup: 161 µs, against 178 µs with the hint on the stores too).
template <typename E, int H>
__global__ __launch_bounds__(256 * H) void gather_kernel(GatherArgs a) {
  constexpr int X = 16 / sizeof(E);
  const int hl = threadIdx.x >> 8, tl = threadIdx.x & 255;
  const int j = blockIdx.x, h = blockIdx.y * H + hl, b = blockIdx.z;
  if (h >= a.Hkv) return;
  const int nch = a.D / X;
  int L = a.ctx[b];
  L = L < 0 ? 0 : L;
  const int lim = L < a.out_len ? L : a.out_len;
  int64_t phys = -1;
  if (j < a.max_blocks && (int64_t)j * a.bs < lim) {
    const int64_t p = a.bt[(int64_t)b * a.max_blocks + j];
    if (p >= 0 && p < a.num_pages) phys = p;
  }
  const int rows = nch * a.bs;
  for (int idx = tl; idx < rows; idx += 256) {
    const int t = idx % a.bs;
    const int c = idx / a.bs;
    const int64_t pos = (int64_t)j * a.bs + t;
    if (pos >= a.out_len) continue;
    const int64_t orow = (((int64_t)b * a.Hkv + h) * a.out_len + pos) * a.D + (int64_t)c * X;
    union {
      Chunk16 c16;
      E e[X];
    } kv, vv;
    kv.c16 = Chunk16{{0u, 0u, 0u, 0u}};
    vv.c16 = Chunk16{{0u, 0u, 0u, 0u}};
    if (phys >= 0 && pos < lim) {
      const int64_t head_base = phys * a.Hkv + h;
      kv.c16 = ld<true, Chunk16>(static_cast<const E*>(a.k_pool) + ((head_base * nch + c) * a.bs + t) * X);
      const E* vb = static_cast<const E*>(a.v_pool) + head_base * a.D * a.bs + (int64_t)c * X * a.bs + t;
#pragma unroll
      for (int i = 0; i < X; ++i) vv.e[i] = vb[(int64_t)i * a.bs];
    }
    st<false, Chunk16>(static_cast<E*>(a.k_out) + orow, kv.c16);
    st<false, Chunk16>(static_cast<E*>(a.v_out) + orow, vv.c16);
  }
}

// The same gather for 2-byte elements on 16-row pages: grid (logical page, group of H kv
// heads, sequence), 2 D threads per kv head.  Thread t of a head takes row t / (D/8) and
// 8-element chunk t % (D/8): its K chunk is one 16-byte load (the K page keeps a row's
// chunk contiguous); the V page ([D][16]) is staged in LDS with one 16-byte load per
// thread and read back as the row's 8 elements of the chunk.  Consecutive threads store
// consecutive chunks of a row, so a wave stores whole output rows.  All loads of a thread
// are issued before the barrier; rows past the context or on an invalid page are stored
// as zeros without loads.  C2's batch: 147 us against 152.5 us for gather_kernel at four
// kv heads per workgroup (lanes along the rows, each V chunk from 8 two-byte loads).
template <int D, int H>
__global__ __launch_bounds__(1024) void gather16_kernel(GatherArgs a) {
  constexpr int NC = D / 8;  // 16-byte chunks per row
  __shared__ Chunk16 s_v[H][2 * D];
  const int hl = threadIdx.x / (2 * D), t = threadIdx.x - hl * (2 * D);
  const int j = blockIdx.x, h = blockIdx.y * H + hl, b = blockIdx.z;
  int L = a.ctx[b];
  L = L < 0 ? 0 : L;
  const int lim = L < a.out_len ? L : a.out_len;
  int64_t phys = -1;
  if (h < a.Hkv && j < a.max_blocks && (int64_t)j * 16 < lim) {
    const int64_t p = a.bt[(int64_t)b * a.max_blocks + j];
    if (p >= 0 && p < a.num_pages) phys = p;
  }
  const int r = t / NC, c = t - r * NC;
  const int64_t pos = (int64_t)j * 16 + r;
  const bool has = phys >= 0 && pos < lim;
  Chunk16 kv = Chunk16{{0u, 0u, 0u, 0u}};
  if (phys >= 0) {  // uniform per kv head
    const int64_t tile = (phys * a.Hkv + h) * (int64_t)(16 * D);  // elements
    s_v[hl][t] = ld<true, Chunk16>(static_cast<const uint16_t*>(a.v_pool) + tile + 8 * t);
    if (has) kv = ld<true, Chunk16>(static_cast<const uint16_t*>(a.k_pool) + tile + (c * 16 + r) * 8);
  }
  __syncthreads();
  if (h >= a.Hkv || pos >= a.out_len) return;
  Chunk16 vv = Chunk16{{0u, 0u, 0u, 0u}};
  if (has) {
    const uint16_t* sv = reinterpret_cast<const uint16_t*>(s_v[hl]);
    uint16_t e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = sv[(8 * c + i) * 16 + r];
    vv = __builtin_bit_cast(Chunk16, e);
  }
  const int64_t orow = (((int64_t)b * a.Hkv + h) * a.out_len + pos) * D + 8 * c;
  st<false, Chunk16>(static_cast<uint16_t*>(a.k_out) + orow, kv);
  st<false, Chunk16>(static_cast<uint16_t*>(a.v_out) + orow, vv);
}

// ---------------------------------------------------------------------------
// index gather / scatter on a contiguous-layout [B][H][S][D] cache
// ---------------------------------------------------------------------------
struct IndexArgs {
  const void* src;
  void* dst;
  int64_t s_b, s_h, s_s, s_d;  // strides of the indexed cache
  int64_t o_b, o_h, o_s, o_d;  // strides of the dense side (gather out / scatter values)
  const int64_t* idx;
  int n_idx, H, S, D;
  int64_t total;
};

// Elements per thread (grid-stride).  On the ops bench's 1024 of 4096 positions (fp16,
// 8 heads, D 128): gather / scatter 25.0 / 25.0 us at 1, 24.6-24.8 / 23.6 us at 2, 26.4 /
// 25.1 us at 4, 28.3 / 26.7 us at 8.
constexpr int kIdxU = 2;

// kIdxU elements per thread, gid + u * (grid threads), in three phases so every load of
// the thread is in flight together: the elements' indices, then their source rows, then
// the stores.  GATHER: out[b,h,j] = kv[b,h,idx[j]] (zero row for an out-of-range index).
// SCATTER: kv[b,h,idx[j]] = values[b,h,j] (out-of-range index skipped).  16-byte stores
// carry the non-temporal hint, and so do the gather's cache reads (the scatter's dense
// reads measured faster without).
template <typename E, bool VEC, bool GATHER>
__global__ __launch_bounds__(256) void index_copy_kernel(IndexArgs a) {
  constexpr int X = VEC ? 16 / (int)sizeof(E) : 1;
  using V = typename std::conditional<VEC, Chunk16, E>::type;
  const int per_row = a.D / X;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int e[kIdxU], jj[kIdxU];
  int64_t bh[kIdxU], ix[kIdxU];
#pragma unroll
  for (int u = 0; u < kIdxU; ++u) {
    const int64_t g = gid + u * stride < a.total ? gid + u * stride : 0;
    e[u] = (int)(g % per_row);
    const int64_t r = g / per_row;
    jj[u] = (int)(r % a.n_idx);
    bh[u] = r / a.n_idx;  // b * H + h
    ix[u] = a.idx[jj[u]];
  }
  int64_t cache_row[kIdxU], dense_row[kIdxU];
  bool ok[kIdxU];
  V val[kIdxU];
#pragma unroll
  for (int u = 0; u < kIdxU; ++u) {
    const int h = (int)(bh[u] % a.H);
    const int64_t b = bh[u] / a.H;
    ok[u] = gid + u * stride < a.total && ix[u] >= 0 && ix[u] < a.S;
    cache_row[u] = b * a.s_b + h * a.s_h + (ok[u] ? ix[u] : 0) * a.s_s + (int64_t)e[u] * X * a.s_d;
    dense_row[u] = b * a.o_b + h * a.o_h + (int64_t)jj[u] * a.o_s + (int64_t)e[u] * X * a.o_d;
    const E* src = static_cast<const E*>(a.src) + (GATHER ? cache_row[u] : dense_row[u]);
    if constexpr (VEC) {
      val[u] = Chunk16{{0u, 0u, 0u, 0u}};
      if (ok[u]) val[u] = GATHER ? ld<true, Chunk16>(src) : ld<false, Chunk16>(src);
    } else {
      val[u] = ok[u] ? *src : E(0);
    }
  }
#pragma unroll
  for (int u = 0; u < kIdxU; ++u) {
    if (gid + u * stride >= a.total) continue;
    if constexpr (GATHER) {
      E* o = static_cast<E*>(a.dst) + dense_row[u];
      if constexpr (VEC) st<true, Chunk16>(o, val[u]);
      else *o = val[u];
    } else {
      if (!ok[u]) continue;
      E* o = static_cast<E*>(a.dst) + cache_row[u];
      if constexpr (VEC) st<true, Chunk16>(o, val[u]);
      else *o = val[u];
    }
  }
}

inline unsigned blocks_for(int64_t total, int per_block) {
  return (unsigned)((total + per_block - 1) / per_block);
}

constexpr int64_t kMaxGrid = 2147483647LL;

// One thread per new token; latency-bound (a few KiB), it takes the place of a host-built
// list and its synchronous copy.
__global__ __launch_bounds__(256) void chunk_slots_kernel(const int32_t* bt, const int32_t* ctx,
                                                          int64_t total, int n, int max_blocks, int bs,
                                                          int32_t* slots) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int64_t b = i / n;
  const int pos = ctx[b] - n + (int)(i - b * n);
  int slot = -1;
  if (pos >= 0 && pos / bs < max_blocks) {
    const int page = bt[b * max_blocks + pos / bs];
    if (page >= 0) slot = page * bs + pos % bs;
  }
  slots[i] = slot;
}

}  // namespace
}  // namespace ivakv

using namespace ivakv;

extern "C" int ivakv_chunk_slots(const int32_t* block_tables, const int32_t* context_lens,
                                 int batch, int n, int max_blocks, int block_size, int32_t* slots,
                                 hipStream_t stream) {
  const char* name = "ivakv_chunk_slots";
  if (batch < 0 || n < 0 || max_blocks < 0 || block_size <= 0)
    return fail(IVAKV_E_ARG, "%s: bad sizes B=%d n=%d max_blocks=%d block_size=%d", name, batch, n,
                max_blocks, block_size);
  const int64_t total = (int64_t)batch * n;
  if (total > (int64_t)1 << 38) return fail(IVAKV_E_SHAPE, "%s: launch too large", name);
  if (total == 0) return IVAKV_OK;
  if (!context_lens || !slots || (max_blocks > 0 && !block_tables))
    return fail(IVAKV_E_ARG, "%s: null pointer argument", name);
  chunk_slots_kernel<<<dim3((unsigned)((total + 255) / 256)), 256, 0, stream>>>(
      block_tables, context_lens, total, n, max_blocks, block_size, slots);
  return launch_status(name);
}

extern "C" int ivakv_append(const void* k_new, const void* v_new, int64_t k_tok_stride,
                            int64_t k_head_stride, int64_t v_tok_stride, int64_t v_head_stride,
                            void* k_pool, void* v_pool, const int32_t* slot_mapping, int n_tok,
                            int num_kv_heads, int head_dim, int block_size, int num_pages,
                            int dtype, hipStream_t stream) {
  const int es = dtype_size(dtype);
  if (es == 0) return fail(IVAKV_E_DTYPE, "ivakv_append: unknown dtype code %d", dtype);
  if (n_tok < 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size <= 0 || num_pages < 0)
    return fail(IVAKV_E_ARG,
                "ivakv_append: bad sizes n_tok=%d Hkv=%d D=%d block_size=%d num_pages=%d", n_tok,
                num_kv_heads, head_dim, block_size, num_pages);
  const int X = 16 / es;
  if (head_dim % X != 0)
    return fail(IVAKV_E_SHAPE, "ivakv_append: head_dim %d must be a multiple of %d", head_dim, X);
  if (n_tok == 0) return IVAKV_OK;
  if (!k_new || !v_new || !k_pool || !v_pool || !slot_mapping)
    return fail(IVAKV_E_ARG, "ivakv_append: null pointer argument");
  if (k_tok_stride < 0 || k_head_stride < 0 || v_tok_stride < 0 || v_head_stride < 0)
    return fail(IVAKV_E_ARG, "ivakv_append: negative stride");
  AppendArgs a{k_new, v_new, k_tok_stride, k_head_stride, v_tok_stride, v_head_stride,
               k_pool, v_pool, slot_mapping, n_tok, num_kv_heads, head_dim, block_size,
               (int64_t)num_pages * block_size};
  const bool vec = aligned16(k_new) && aligned16(v_new) && aligned16(k_pool) && aligned16(v_pool) &&
                   (k_tok_stride % X == 0) && (k_head_stride % X == 0) &&
                   (v_tok_stride % X == 0) && (v_head_stride % X == 0);
  const int64_t lanes_per_head_group = (int64_t)cdiv(n_tok, 16) * 16 * (head_dim / X);
  const bool few = vec && lanes_per_head_group * cdiv(num_kv_heads, kAppendHeads) < kFewAppendThreads;
  const int64_t per_tok = vec && !few ? (int64_t)cdiv(num_kv_heads, kAppendHeads) : num_kv_heads;
  const int64_t total = lanes_per_head_group * per_tok;
  const int threads = few ? 64 : 256;
  const unsigned grid = blocks_for(total, threads);
  if ((int64_t)grid > kMaxGrid) return fail(IVAKV_E_SHAPE, "ivakv_append: too many rows");
  const int64_t elems = (int64_t)n_tok * num_kv_heads * head_dim;
  const int scale = head_dim == 256 ? 4 : 1;
  if (es == 2 && vec && block_size == 16 && (head_dim == 64 || head_dim == 128 || head_dim == 256) &&
      n_tok >= scale * kRunTokens && elems >= scale * kRunElems) {
    const int64_t wgs = (int64_t)cdiv(n_tok, 16) * cdiv(num_kv_heads, 4);
    if (wgs > kMaxGrid) return fail(IVAKV_E_SHAPE, "ivakv_append: too many rows");
    const dim3 rg((unsigned)wgs);
    if (head_dim == 64) append_runs_kernel<64><<<rg, 256, 0, stream>>>(a);
    else if (head_dim == 128) append_runs_kernel<128><<<rg, 256, 0, stream>>>(a);
    else append_runs_kernel<256><<<rg, 256, 0, stream>>>(a);
    return launch_status("ivakv_append");
  }
  if (es == 4) {
    if (few) append_vec_kernel<uint32_t, 1><<<grid, threads, 0, stream>>>(a);
    else if (vec) append_vec_kernel<uint32_t, kAppendHeads><<<grid, threads, 0, stream>>>(a);
    else append_kernel<uint32_t><<<grid, threads, 0, stream>>>(a);
  } else {
    if (few) append_vec_kernel<uint16_t, 1><<<grid, threads, 0, stream>>>(a);
    else if (vec) append_vec_kernel<uint16_t, kAppendHeads><<<grid, threads, 0, stream>>>(a);
    else append_kernel<uint16_t><<<grid, threads, 0, stream>>>(a);
  }
  return launch_status("ivakv_append");
}

// kv heads per workgroup of the gather (C2 batch: 1 / 2 / 4 heads 161 / 156.5 / 152.5 us)
constexpr int kGatherHeads = 4;

extern "C" int ivakv_gather(const void* k_pool, const void* v_pool, const int32_t* block_tables,
                            const int32_t* context_lens, int batch, int max_blocks,
                            int num_kv_heads, int head_dim, int block_size, int num_pages,
                            int out_len, void* k_out, void* v_out, int dtype,
                            hipStream_t stream) {
  const int es = dtype_size(dtype);
  if (es == 0) return fail(IVAKV_E_DTYPE, "ivakv_gather: unknown dtype code %d", dtype);
  if (batch < 0 || max_blocks < 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size <= 0 ||
      num_pages < 0 || out_len < 0)
    return fail(IVAKV_E_ARG,
                "ivakv_gather: bad sizes B=%d max_blocks=%d Hkv=%d D=%d block_size=%d "
                "num_pages=%d out_len=%d",
                batch, max_blocks, num_kv_heads, head_dim, block_size, num_pages, out_len);
  const int X = 16 / es;
  if (head_dim % X != 0)
    return fail(IVAKV_E_SHAPE, "ivakv_gather: head_dim %d must be a multiple of %d", head_dim, X);
  if (batch == 0 || out_len == 0) return IVAKV_OK;
  if (!k_pool || !v_pool || !context_lens || !k_out || !v_out || (max_blocks > 0 && !block_tables))
    return fail(IVAKV_E_ARG, "ivakv_gather: null pointer argument");
  if (!aligned16(k_pool) || !aligned16(v_pool) || !aligned16(k_out) || !aligned16(v_out))
    return fail(IVAKV_E_ARG, "ivakv_gather: pools and outputs must be 16-byte aligned");
  if (batch > 65535 || num_kv_heads > 65535)
    return fail(IVAKV_E_SHAPE, "ivakv_gather: batch and num_kv_heads must be <= 65535");
  GatherArgs a{k_pool, v_pool, block_tables, context_lens, max_blocks, num_kv_heads, head_dim,
               block_size, num_pages, out_len, k_out, v_out};
  if (es == 2 && block_size == 16 && (head_dim == 64 || head_dim == 128 || head_dim == 256)) {
    // 1024 threads: 2 D per kv head
    const int hpw = 512 / head_dim;
    const dim3 g16((unsigned)cdiv(out_len, 16), (unsigned)cdiv(num_kv_heads, hpw), (unsigned)batch);
    switch (head_dim) {
      case 64: gather16_kernel<64, 8><<<g16, 1024, 0, stream>>>(a); break;
      case 128: gather16_kernel<128, 4><<<g16, 1024, 0, stream>>>(a); break;
      default: gather16_kernel<256, 2><<<g16, 1024, 0, stream>>>(a); break;
    }
    return launch_status("ivakv_gather");
  }
  constexpr int kH = kGatherHeads;
  dim3 grid((unsigned)cdiv(out_len, block_size), (unsigned)cdiv(num_kv_heads, kH), (unsigned)batch);
  if (es == 4) gather_kernel<uint32_t, kH><<<grid, 256 * kH, 0, stream>>>(a);
  else gather_kernel<uint16_t, kH><<<grid, 256 * kH, 0, stream>>>(a);
  return launch_status("ivakv_gather");
}

namespace {

int index_copy(bool gather, const char* name, const void* src, void* dst, int64_t s_b, int64_t s_h,
               int64_t s_s, int64_t s_d, int64_t o_b, int64_t o_h, int64_t o_s, int64_t o_d,
               const int64_t* indices, int n_idx, int batch, int n_heads, int seq_len,
               int head_dim, int dtype, hipStream_t stream) {
  const int es = dtype_size(dtype);
  if (es == 0) return fail(IVAKV_E_DTYPE, "%s: unknown dtype code %d", name, dtype);
  if (n_idx < 0 || batch < 0 || n_heads < 0 || seq_len < 0 || head_dim < 0)
    return fail(IVAKV_E_ARG, "%s: negative size", name);
  const int64_t rows = (int64_t)batch * n_heads * n_idx;
  if (rows == 0 || head_dim == 0) return IVAKV_OK;
  if (!src || !dst || !indices) return fail(IVAKV_E_ARG, "%s: null pointer argument", name);
  const int X = 16 / es;
  const bool vec = s_d == 1 && o_d == 1 && head_dim % X == 0 && aligned16(src) && aligned16(dst) &&
                   s_b % X == 0 && s_h % X == 0 && s_s % X == 0 && o_b % X == 0 &&
                   o_h % X == 0 && o_s % X == 0;
  IndexArgs a{src, dst, s_b, s_h, s_s, s_d, o_b, o_h, o_s, o_d, indices, n_idx, n_heads, seq_len,
              head_dim, rows * (vec ? head_dim / X : head_dim)};
  const unsigned grid = blocks_for((a.total + kIdxU - 1) / kIdxU, 256);
  if ((int64_t)grid > kMaxGrid) return fail(IVAKV_E_SHAPE, "%s: too many rows", name);
#define IVAKV_IDX_LAUNCH(E)                                                              \
  do {                                                                                   \
    if (gather) {                                                                        \
      if (vec) index_copy_kernel<E, true, true><<<grid, 256, 0, stream>>>(a);            \
      else index_copy_kernel<E, false, true><<<grid, 256, 0, stream>>>(a);               \
    } else {                                                                             \
      if (vec) index_copy_kernel<E, true, false><<<grid, 256, 0, stream>>>(a);           \
      else index_copy_kernel<E, false, false><<<grid, 256, 0, stream>>>(a);              \
    }                                                                                    \
  } while (0)
  if (es == 4) IVAKV_IDX_LAUNCH(uint32_t);
  else IVAKV_IDX_LAUNCH(uint16_t);
#undef IVAKV_IDX_LAUNCH
  return launch_status(name);
}

}  // namespace

extern "C" int ivakv_index_gather(const void* kv, int64_t s_b, int64_t s_h, int64_t s_s,
                                  int64_t s_d, const int64_t* indices, int n_idx, int batch,
                                  int n_heads, int seq_len, int head_dim, void* out, int dtype,
                                  hipStream_t stream) {
  const int64_t o_s = head_dim, o_h = (int64_t)n_idx * head_dim, o_b = (int64_t)n_heads * o_h;
  return index_copy(true, "ivakv_index_gather", kv, out, s_b, s_h, s_s, s_d, o_b, o_h, o_s, 1,
                    indices, n_idx, batch, n_heads, seq_len, head_dim, dtype, stream);
}

extern "C" int ivakv_index_scatter(void* kv, int64_t s_b, int64_t s_h, int64_t s_s, int64_t s_d,
                                   const int64_t* indices, int n_idx, const void* values,
                                   int64_t v_b, int64_t v_h, int64_t v_s, int64_t v_d, int batch,
                                   int n_heads, int seq_len, int head_dim, int dtype,
                                   hipStream_t stream) {
  return index_copy(false, "ivakv_index_scatter", values, kv, s_b, s_h, s_s, s_d, v_b, v_h, v_s,
                    v_d, indices, n_idx, batch, n_heads, seq_len, head_dim, dtype, stream);
}
