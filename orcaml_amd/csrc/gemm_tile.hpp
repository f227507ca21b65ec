// Small-tile fp32 MFMA product kernel (part of gemm.hip, which defines
// GemmParams, floatx16 and write_tile): T x T tiles of C for T = 16, 32 or 64.
//
// What bounds the products it takes is latency and the number of CUs at work,
// not the matrix cores: a 64 x 128 x 784 product is one 128 x 128 tile, whose
// 25 slabs keep one CU's MFMA pipes busy for 43 us, but 32 tiles of 16 x 16.
// A block is four waves and a slab of KS = 4096 / T k-values (16 KiB of each
// operand, four float4 per thread and operand whatever T is), so the layout of
// a load is the same work per thread in every form:
//   T = 16  four waves split the slab's k range (64 each, v_mfma_f32_16x16x4f32)
//   T = 32  four waves split it too (32 each, v_mfma_f32_32x32x2f32)
//   T = 64  2 x 2 waves, each a 32 x 32 block over the whole slab
// A wave sums its even and odd MFMA steps apart (two independent chains).  The
// split forms add their four waves' blocks in wave order through LDS.
//
// Slabs come through slab.hpp's loader and loop.

// One element's epilogue (C at [m][n] gets v).
__device__ __forceinline__ void tile_store_one(const GemmParams& p, float* C, int64_t ldc, int epi, int m, int n, float v) {
  switch (epi) {
    case ORCA_HIP_EPI_BIAS: v = v + p.bias[n]; break;
    case ORCA_HIP_EPI_BIAS_RELU:
      v = v + p.bias[n];
      v = v > 0.0f ? v : 0.0f;
      break;
    case ORCA_HIP_EPI_RELU_MASK: v = p.mask[(int64_t)m * p.ldmask + n] > 0.0f ? v : 0.0f; break;
    case ORCA_HIP_EPI_BIAS_RELU_PRE:
      v = v + p.bias[n];
      p.pre[(int64_t)m * ldc + n] = v;
      v = v > 0.0f ? v : 0.0f;
      break;
    case ORCA_HIP_EPI_RELU_MASK_PRE:
      p.pre[(int64_t)m * ldc + n] = v;
      v = p.mask[(int64_t)m * p.ldmask + n] > 0.0f ? v : 0.0f;
      break;
    default: break;
  }
  C[(int64_t)m * ldc + n] = v;
}

// Grid (N tiles, M tiles [+ 1], batch * splits).  The extra row of blocks, when
// p.colsum is set (row-major B, one batch entry), takes B's column sums over the
// whole K range: a block's first T threads add their column's values in
// ascending k from +0 out of the same LDS slabs (the additions of sum_to_shape,
// so the same bits), beside the product instead of in a launch after it.
// ONE: K is at most one slab.  Without the loop and its second buffer four blocks fit a CU
// instead of two, so that some load or store while others multiply, and the code is a
// third as long.
template <int T, bool TA, bool TB, bool UA>
constexpr int tile_slab_floats() {
  return TileOperand<T, !TA, UA>::FLOATS + TileOperand<T, TB, UA>::FLOATS;
}

struct NoUpdate {
  static constexpr bool used = false;
  template <int E>
  struct State {};
  template <int E>
  __device__ __forceinline__ void load(State<E>&, int, size_t) const {}
};

// U: what becomes of an element of C and of a column sum besides being stored (NoUpdate, or
// TileUpdate below; whole products without an epilogue only).
template <int T, bool TA, bool TB, bool UA, bool ONE, class U = NoUpdate>
__device__ __forceinline__ void tile_product(const GemmParams& p, int bx, int by, int bz, float* __restrict__ smem,
                                             const U& upd = U()) {
  using OpA = TileOperand<T, !TA, UA>;
  using OpB = TileOperand<T, TB, UA>;
  constexpr int KS = OpA::KS;
  constexpr int SLAB = tile_slab_floats<T, TA, TB, UA>();
  static_assert(SLAB >= (T == 64 ? 0 : 4 * T * T), "the waves' blocks fit a slab buffer");

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int n0 = bx * T, m0 = by * T;
  const int batch = bz / p.splits, split = bz % p.splits;
  floatx4 sa[2][4], sb[2][4];  // the register stages

  if (!TB && m0 >= p.M) {  // the column sums
    if (bz) return;
    OpB ob;
    ob.init(p.B, p.ldb, n0, p.N, 0, p.K, p.K);
    float cs = 0.0f;
    slab_pipeline<ONE>(
        (p.K + KS - 1) / KS, [&](int t, auto st) { ob.load(t, sb[decltype(st)::value]); },
        [&](int t, auto st, auto buf, auto last) {
          ob.template store<decltype(last)::value>(t, sb[decltype(st)::value], smem + decltype(buf)::value * SLAB);
        },
        []() {},
        [&](int t, auto buf, auto mid, bool more, auto) {
          mid();
          if (tid < T) {
            const float* s = smem + decltype(buf)::value * SLAB + tid;
            const int rows = min(KS, p.K - t * KS);
            // 64 rows' reads ahead of their adds (rows past K are zero): the chain of adds
            // is what takes the time, 4.6 to 5.5 ns a row with the loads (X^T dY of 16 x 112 x 1288:
            // 9.3 us beside a product of 6.1), 6.6 where T is 32 or 64
            for (int k = 0; k < rows; k += 64) {
              float v[64];
#pragma unroll
              for (int q = 0; q < 64; ++q) v[q] = s[OpB::mn_off(k + q)];
#pragma unroll
              for (int q = 0; q < 64; ++q) cs = cs + v[q];
            }
          }
          if (more) __syncthreads();
        });
    if (tid < T && n0 + tid < p.N) {
      p.colsum[n0 + tid] = cs;
      if constexpr (U::used) upd.bias(n0 + tid, cs);
    }
    return;
  }

  const int kb = split * p.k_chunk, kend = min(p.K, kb + p.k_chunk);
  const int n = (kend - kb + KS - 1) / KS;
  OpA oa;
  OpB ob;
  oa.init(p.A + batch * p.sa, p.lda, m0, p.M, kb, kend, p.K);
  ob.init(p.B + batch * p.sb, p.ldb, n0, p.N, kb, kend, p.K);

  constexpr int LW = T == 16 ? 16 : 32;  // lanes of one k group
  const int i = lane % LW, g = lane / LW;
  const int ra = T == 64 ? (wave >> 1) * 32 + i : i, rb = T == 64 ? (wave & 1) * 32 + i : i;
  const int kw = T == 64 ? 16 * g : wave * (KS / 4) + 16 * g;

  using Acc = typename std::conditional<T == 16, floatx4, floatx16>::type;
  Acc acc[2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int r = 0; r < (T == 16 ? 4 : 16); ++r) acc[c][r] = 0.0f;

  // An updated element's state is loaded before the product where that is a few registers.
  constexpr int NU = T == 64 ? 16 : T * T / 256;  // elements per thread
  [[maybe_unused]] typename U::template State<NU> us;
  [[maybe_unused]] const int u_row = T == 64 ? m0 + (wave >> 1) * 32 + g * 4 : m0 + tid / T, u_col = T == 64 ? n0 + rb : n0 + tid % T;
  [[maybe_unused]] auto row_of = [&](int e) { return T == 64 ? u_row + (e >> 2) * 8 + (e & 3) : u_row + 256 / T * e; };
  [[maybe_unused]] auto load_update = [&]() {
#pragma unroll
    for (int e = 0; e < NU; ++e)
      upd.load(us, e, (size_t)min(row_of(e), p.M - 1) * p.ldc + min(u_col, p.N - 1));
  };
  if constexpr (U::used && T < 64) load_update();

  constexpr int HS = T == 64 ? 16 : 8;  // MFMA steps in half a slab
  float fa[2][HS], fb[2][HS];
  auto frags = [&](const float* s, int half, float (&a)[HS], float (&b)[HS]) {
    OpA::frag(s, ra, kw + (T == 64 ? 32 : 8) * half, a);
    OpB::frag(s + OpA::FLOATS, rb, kw + (T == 64 ? 32 : 8) * half, b);
  };
  auto mfma = [&](const float (&a)[HS], const float (&b)[HS]) {
#pragma unroll
    for (int q = 0; q < HS; ++q) {
      if constexpr (T == 16)
        acc[q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], b[q], acc[q & 1], 0, 0, 0);
      else
        acc[q & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q], b[q], acc[q & 1], 0, 0, 0);
    }
  };
  // Memory instructions placed among the matrix instructions: per half slab RD fragment
  // reads, and in the first half eight LDS stores and eight loads.
  constexpr int RD = (!TA ? HS / 4 : HS / 2) + (TB ? HS / 4 : HS / 2);
  auto interleave = [&](auto first) {
#pragma unroll
    for (int q = 0; q < HS; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
      if (q < RD) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
      if (decltype(first)::value && q % (HS / 8) == 0) {
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // DS write
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // VMEM read
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  slab_pipeline<ONE>(
      n,
      [&](int t, auto st) {
        oa.load(t, sa[decltype(st)::value]);
        ob.load(t, sb[decltype(st)::value]);
      },
      [&](int t, auto st, auto buf, auto last) {
        float* s = smem + decltype(buf)::value * SLAB;
        oa.template store<decltype(last)::value>(t, sa[decltype(st)::value], s);
        ob.template store<decltype(last)::value>(t, sb[decltype(st)::value], s + OpA::FLOATS);
      },
      [&]() { frags(smem, 0, fa[0], fb[0]); },
      [&](int, auto buf, auto mid, bool more, auto full) {
        // the second half's fragments, the store and the loads go under the first half's
        // multiplications, the barrier and the next slab's first fragments under the second's
        constexpr int P = decltype(buf)::value;
        frags(smem + P * SLAB, 1, fa[1], fb[1]);
        mid();
        mfma(fa[0], fb[0]);
        if constexpr (decltype(full)::value) interleave(std::true_type{});
        if (!ONE && more) {
          __syncthreads();
          frags(smem + (P ^ 1) * SLAB, 0, fa[0], fb[0]);
        }
        // a K up to 32 is in the first half of a one-slab 64-tile; the other would multiply zeros,
        // 0.43 us of each wave (X^T dY of 2183 x 832 x 8: 6.3 -> 5.4 us, 2048 x 2048 x 32: 9.6 -> 7.9)
        if (!(ONE && T == 64) || p.K > 32) mfma(fa[1], fb[1]);
        if constexpr (decltype(full)::value) interleave(std::false_type{});
      });

  float* C = p.C + batch * p.sc;
  if (p.splits > 1) C = p.C + (int64_t)bz * p.M * p.N;
  const int64_t ldc = p.splits > 1 ? p.N : p.ldc;
  const int epi = p.splits > 1 ? ORCA_HIP_EPI_NONE : p.epi;
  if constexpr (T == 64) {
    floatx16 sum[1][1];
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[0][0][r] = acc[0][r] + acc[1][r];
    if constexpr (U::used) {
      load_update();
#pragma unroll
      for (int e = 0; e < NU; ++e)
        if (row_of(e) < p.M && u_col < p.N) upd.store(us, e, (size_t)row_of(e) * p.ldc + u_col, sum[0][0][e]);
      return;
    }
    write_tile(sum, C, ldc, epi, m0 + (wave >> 1) * 32, n0 + (wave & 1) * 32, m0 + T <= p.M && n0 + T <= p.N, p);
  } else {
    __syncthreads();  // the last slab's fragments are read
    float* red = smem + wave * T * T;
#pragma unroll
    for (int r = 0; r < (T == 16 ? 4 : 16); ++r) {
      const int row = T == 16 ? g * 4 + r : (r >> 2) * 8 + g * 4 + (r & 3);
      red[row * T + i] = acc[0][r] + acc[1][r];
    }
    __syncthreads();
    // element e of thread t: row t / T + e * 256 / T, column t % T
    const int col = n0 + tid % T;
#pragma unroll
    for (int e = 0; e < T * T / 256; ++e) {
      const int o = tid + 256 * e;
      const int row = m0 + o / T;
      const float v = ((smem[o] + smem[o + T * T]) + smem[o + 2 * T * T]) + smem[o + 3 * T * T];
      if (row < p.M && col < p.N) {
        if constexpr (U::used)
          upd.store(us, e, (size_t)row * p.ldc + col, v);
        else
          tile_store_one(p, C, ldc, epi, row, col, v);
      }
    }
  }
}

template <int T, bool TA, bool TB, bool UA, bool ONE>
__global__ void __launch_bounds__(256, ONE ? 4 : 2) gemm_tile_kernel(GemmParams p) {
  __shared__ __attribute__((aligned(16))) float smem[(ONE ? 1 : 2) * tile_slab_floats<T, TA, TB, UA>()];
  // the column sums' chain of adds starts first
  const int by = TB || !p.colsum ? blockIdx.y : blockIdx.y ? blockIdx.y - 1 : (p.M + T - 1) / T;
  tile_product<T, TA, TB, UA, ONE>(p, blockIdx.x, by, blockIdx.z, smem);
}

// The same for a batched product on 64 x 64 tiles.  Consecutive workgroups go round the eight
// XCDs, each with its own L2; here an XCD takes one run of consecutive tiles instead, so that
// the tiles of a batch entry, which share its operands, read them through one L2: 96 x [197 x
// 64] x [64 x 197] and both gradients 50.2 -> 46.8 us, 32 x [512 x 64] x [64 x 512] 47.2 ->
// 44.4.  (Entries of smaller tiles: no difference.  A single product keeps the dispatch order,
// in which an XCD has every eighth column of tiles with all of its rows, and a kernel without
// this arithmetic: as a branch of one kernel it cost single products 0.2 us a launch.)
// Batched products have no epilogue: without the others' code 46.8 -> 43.0 us.
template <bool TA, bool TB, bool UA, bool ONE>
__global__ void __launch_bounds__(256, ONE ? 4 : 2) gemm_tile_batch_kernel(GemmParams p) {
  __shared__ __attribute__((aligned(16))) float smem[(ONE ? 1 : 2) * tile_slab_floats<64, TA, TB, UA>()];
  const uint32_t nx = gridDim.x, per = nx * gridDim.y, blocks = per * gridDim.z;
  const uint32_t l = blockIdx.x + nx * blockIdx.y + per * blockIdx.z, xcd = l % 8;
  const uint32_t id = xcd * (blocks / 8) + min(xcd, blocks % 8) + l / 8, in = id % per;
  p.epi = ORCA_HIP_EPI_NONE;
  tile_product<64, TA, TB, UA, ONE>(p, in % nx, in / nx, id / per, smem);
}

// A Linear layer's two backward products from one grid: the column sums of dW = X^T dY (w;
// w_sums blocks, none without them), dX = dY W^T (x; x_blocks, x_nt of them per row of tiles)
// and dW itself.  Neither
// fills the GPU at the sizes that come here, and each launch of its own pays the start and
// the drain of a grid again.
template <int TX, int TW, bool UA>
__global__ void __launch_bounds__(256, 2) gemm_tile_pair_kernel(GemmParams x, GemmParams w, int w_sums, int x_blocks, int x_nt, int w_nt) {
  constexpr int SX = tile_slab_floats<TX, false, true, UA>(), SW = tile_slab_floats<TW, true, false, UA>();
  __shared__ __attribute__((aligned(16))) float smem[2 * (SX > SW ? SX : SW)];
  const int b = (int)blockIdx.x - w_sums, c = b - x_blocks;
  if (b >= 0 && c < 0) {
    tile_product<TX, false, true, UA, false>(x, b % x_nt, b / x_nt, 0, smem);
  } else {
    const int by = b < 0 ? (w.M + TW - 1) / TW : c / w_nt;
    tile_product<TW, true, false, UA, false>(w, b < 0 ? (int)blockIdx.x : c % w_nt, by, 0, smem);
  }
}

// A model's whole optimizer step in the launch of its last product, dW of layer 0: column sums
// (w_sums blocks), dW's tiles (w_blocks), whose blocks update the elements that they produce,
// and the rest of the arenas, elements [rest, u.n), 4096 a block.  Nothing else of the step
// reads W_0, and dW reads no parameter, so the update needs no pass of its own: its memory
// traffic runs beside the product, W_0's gradient is not read back, and the launch with its
// start and drain goes.  Same arithmetic per element as the passes in fused.hip, same bits.
// 64 SGD steps of 784-128-128-10 / B 64 with a read 2219 -> 2084 us, 32 AdamW steps of
// 784-1024-1024-10 / B 256 2820 -> 2753 us and of 500-1001-333-26 / B 200 2558 -> 2441 us.
template <bool ADAMW>
struct TileUpdate {
  static constexpr bool used = true;
  template <int E>
  struct State {
    float p[E], m[E], v[E];
  };
  const ArenaUpdate& u;
  const AdamWScalars& k;
  size_t b0;  // the bias's first element

  template <int E>
  __device__ __forceinline__ void load(State<E>& s, int e, size_t i) const {
    s.p[e] = u.P[i];
    if (ADAMW) {
      s.m[e] = u.M[i];
      s.v[e] = u.V[i];
    }
  }
  template <int E>
  __device__ __forceinline__ void store(State<E>& s, int e, size_t i, float g) const {
    u.G[i] = g;
    if (ADAMW) {
      adamw_elem(s.p[e], g, s.m[e], s.v[e], k);
      u.M[i] = s.m[e];
      u.V[i] = s.v[e];
      u.P[i] = s.p[e];
    } else {
      u.P[i] = s.p[e] - g * k.lr;
    }
  }
  __device__ __forceinline__ void bias(int c, float g) const {
    State<1> s;
    load(s, 0, b0 + c);
    store(s, 0, b0 + c, g);
  }
};

constexpr int kUpdateBlock = 4096;  // arena elements per updating block: four float4 of each array per thread

template <int T, bool UA, bool ONE, bool ADAMW>
__global__ void __launch_bounds__(256, ONE ? 4 : 2)
    gemm_tile_update_kernel(GemmParams w, ArenaUpdate u, int w_sums, int w_blocks, int w_nt, size_t bias, size_t rest) {
  __shared__ __attribute__((aligned(16))) float smem[(ONE ? 1 : 2) * tile_slab_floats<T, true, false, UA>()];
  const AdamWScalars k = u.kdev ? *u.kdev : u.k;
  const int b = (int)blockIdx.x - w_sums, c = b - w_blocks;
  if (c < 0) {
    const int by = b < 0 ? (w.M + T - 1) / T : b / w_nt;
    tile_product<T, true, false, UA, ONE>(w, b < 0 ? (int)blockIdx.x : b % w_nt, by, 0, smem,
                                          TileUpdate<ADAMW>{u, k, bias});
    return;
  }
  // arena offsets are multiples of 64 elements, so every group of four is whole
  const size_t i0 = rest + (size_t)c * kUpdateBlock + threadIdx.x * 4;
  floatx4 p[4], g[4], m[4], v[4];
  auto ld = [&](const float* a, int j) {
    return __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(a + min(i0 + 1024 * j, u.n - 4)));
  };
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    p[j] = ld(u.P, j);
    g[j] = ld(u.G, j);
    if (ADAMW) {
      m[j] = ld(u.M, j);
      v[j] = ld(u.V, j);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const size_t i = i0 + 1024 * j;
    if (i >= u.n) return;
    auto st = [&](float* a, floatx4 x) { __builtin_nontemporal_store(x, reinterpret_cast<floatx4*>(a + i)); };
    if (ADAMW) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float pe = p[j][e], me = m[j][e], ve = v[j][e];
        adamw_elem(pe, g[j][e], me, ve, k);
        p[j][e] = pe;
        m[j][e] = me;
        v[j][e] = ve;
      }
      st(u.M, m[j]);
      st(u.V, v[j]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) p[j][e] = p[j][e] - g[j][e] * k.lr;
    }
    st(u.P, p[j]);
  }
}
