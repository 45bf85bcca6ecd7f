// f32 attention on bf16 matrix products; included by attention.hip (inside
// its namespaces, after attn_body).
//
// Q, K, V and the probabilities are split exactly into three bf16 values each
// and six products are formed per term, as in gemm_f32.hpp; the maximum, the
// exponentials and the sums stay in f32.  A score sums its hi x hi products
// and its small ones in two chains; each 32-key step of P V starts from zero
// and joins O with one fused multiply-add (the f32 MFMA kernel rounds O once
// per four keys).
//
// A work-group owns 64 query rows of one head, 16 per wave, and two groups of
// four waves share their keys: group g takes the 32-key tiles g, g + 2, ...,
// and the groups' (maximum, sum, O) meet in LDS at the end.  Splitting a tile
// is vector work and multiplying it matrix work, and a wave does one after
// the other, so the groups run one phase apart: while one splits K or V into
// its LDS planes (48 KiB, K and V in turn), the other multiplies.
//
// The scores are computed transposed (S^T = K Q^T): a lane holds 8 keys of one
// query.  Tile t, row r of S^T is key 8 (r / 4) + 4 t + r % 4 of the 32, so
// these are the 8 consecutive keys of its B fragment of O^T = V^T P^T, and P
// goes from the softmax into the products without passing LDS.
//
// The split errs by up to 2^-124 for values below 2^-100.  With keys and queries
// below 2^90 that moves a score by less than 2^-26; it moves an output of 2^-97
// or more by less than 2^-27 of itself.  (Probabilities below 2^-100 of the row's
// largest are held to 2^-124 too.)  A query is formed again by attn_body, at the
// end, if it or a key it sees is larger, or if one of its outputs is not finite
// or, with a value below 2^-100 in sight, smaller: that follows from the query
// and what it sees, not from those that share its tile.  777 queries behind 256
// keys, 16 heads x 256 (us; f32 MFMA kernel 227, here 124): a value below 2^-100
// in one key or value row 124; a column of V wholly below 377, an infinity that
// half of the queries see 366, one NaN query 155.
//
// What bounds it: LDS.  A fragment of three planes feeds six products, so with
// 16 queries per wave a key tile reads as many LDS cycles as it multiplies,
// plus the planes' stores; 32 queries per wave would halve that but need twice
// the O registers (64 of 256 now).  16 heads, d = 256, us on the f32 MFMA ->
// here: 777 queries behind 256 keys 230 -> 124, 200 alone 63.9 -> 35.4, 2048
// 461 -> 260, 4096 1694 -> 927; d = 128, 300 behind 31 (4 heads) 47.5 -> 29.4.
// Error against 64 bits (2-norm) 6.9e-7 -> 2.3e-7 at 777 behind 256.

// the six products of a term: planes of the A and B operand, small ones first
constexpr int kPA[6] = {2, 0, 1, 1, 0, 0}, kPB[6] = {0, 2, 1, 0, 1, 0};

template <int D>
__global__ __launch_bounds__(512, 2) void attn_f32_split(AttnParams p) {
  constexpr int BQ = 64, BK = 32;
  constexpr int NKB = D / 32;              // 32-deep k-steps of a score
  constexpr int NDT = D / 16;              // 16-row tiles of O^T
  constexpr int CPR = D / 8;               // 8-element chunks of a key row
  constexpr int CH = BK * CPR / 256;       // chunks per thread and operand
  constexpr int kPlane = BK * D;           // bf16 of a plane (K [32][D], V^T [D][32])
  constexpr int kGroup = 3 * kPlane;
  constexpr int kMerge = 4 * 64 * (NDT * 4 + 2) * 4;  // O, m, l of a group
  constexpr int kTiles = 2 * kGroup * 2;               // bytes of both groups' planes
  constexpr int kQ = 2 * 4 * NKB * 64 * 16;            // the mid and lo planes of Q, by wave row and lane
  constexpr int kMax = kTiles + kQ > kMerge ? kTiles + kQ : kMerge;
  constexpr int kLds = attn_lds_bytes<float, D>() > kMax ? attn_lds_bytes<float, D>() : kMax;
  static_assert(BK * CPR % 256 == 0, "whole chunks per thread");
  static_assert(kLds <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(16))) char smem[kLds];
  // once Q is no longer read: the first large key, the first with a tiny value,
  // and the rows to form again, 16 per wave of group 0
  int* const flags = reinterpret_cast<int*>(smem + kTiles + kQ) - 6;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2, wq = wave & 3, gt = tid & 255;
  const int n = lane & 15, g = lane >> 4;

  const int qtiles = (p.qn + BQ - 1) / BQ;
  // (pinned to scalar registers: the divisions run on vector ones, and a
  // resource based on them would be read lane by lane)
  const int h = __builtin_amdgcn_readfirstlane(blockIdx.x % p.heads);
  const int q0 = __builtin_amdgcn_readfirstlane((qtiles - 1 - static_cast<int>(blockIdx.x / p.heads)) * BQ);  // longest first
  const int kvh = __builtin_amdgcn_readfirstlane(h / (p.heads / p.kvh));
  const int offset = p.kn - p.qn;
  const float* Q = static_cast<const float*>(p.q) + (int64_t)h * p.ldq * D;
  const float* K = static_cast<const float*>(p.k) + (int64_t)kvh * p.ldk * D;
  const float* V = static_cast<const float*>(p.vt) + (int64_t)kvh * D * p.ldv;

  constexpr float kSmallOut = 0x1p-97f;
  constexpr uint32_t kLarge = 217u << 24, kTiny = 27u << 24;  // 2 * bits of 2^90 and 2^-100
  auto largest = [](uint32_t m, const float4_t& a, const float4_t& b) {  // of 2 * bits
#pragma unroll
    for (int e = 0; e < 4; ++e) m = max(max(m, 2u * __float_as_uint(a[e])), 2u * __float_as_uint(b[e]));
    return m;
  };
  auto least = [](uint32_t m, const float4_t& a, const float4_t& b) {  // of 2 * bits - 1 (0 last)
#pragma unroll
    for (int e = 0; e < 4; ++e) m = min(min(m, 2u * __float_as_uint(a[e]) - 1u), 2u * __float_as_uint(b[e]) - 1u);
    return m;
  };
  constexpr int kNone = 0x7fffffff;
  auto wave_least = [](int x) {
    for (int o = 1; o < 64; o <<= 1) x = min(x, __shfl_xor(x, o, 64));
    return __builtin_amdgcn_readfirstlane(x);
  };
  int first_large = kNone, first_tiny = kNone;  // keys, of those that this wave split

  // Q fragments (B operand): d = 32 kb + 8 g .. + 7 of query n; the mid and lo
  // planes, half of the products, wait in LDS (both groups use the same rows;
  // in registers they spill, and a reload waits for the prefetch as well)
  bf16x8 qf[NKB];
  bf16x8* const qml = reinterpret_cast<bf16x8*>(smem + kTiles) + wq * NKB * 128 + lane;
  uint64_t large_q;  // by lane
  {
    uint32_t q_large = 0;
    const float* row = Q + (int64_t)min(q0 + 16 * wq + n, p.qn - 1) * D + 8 * g;
    float4_t raw[NKB][2];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int u = 0; u < 2; ++u) raw[kb][u] = *reinterpret_cast<const float4_t*>(row + 32 * kb + 4 * u);
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      bf16x8 pl[3];
      split8(raw[kb][0], raw[kb][1], pl[0], pl[1], pl[2]);
      q_large = largest(q_large, raw[kb][0], raw[kb][1]);
      qf[kb] = pl[0];
      if (grp == 0) {  // published by the first phase's barrier
        qml[kb * 128] = pl[1];
        qml[kb * 128 + 64] = pl[2];
      }
    }
    large_q = __ballot(q_large >= kLarge);
  }

  // one register set holds the next operand to be split: V of a tile is
  // requested once its K is in LDS, the next K once V is
  float4_t ld[CH][2];
  __bf16* const planes = reinterpret_cast<__bf16*>(smem) + grp * kGroup;
  // chunk i of a thread: K row gt / CPR + i 256 / CPR, V^T row gt / 4 + 64 i
  // (buffer resources: one lane offset each, the rest is uniform)
  auto rsrc = [](const float* base, int64_t n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, static_cast<int>(static_cast<uint32_t>(n * 4)),
                                             0x00020000);
  };
  const __amdgpu_buffer_rsrc_t rK = rsrc(K, (int64_t)p.kn * D), rV = rsrc(V, (int64_t)D * p.ldv);
  const int kr0 = gt / CPR, kc0 = 8 * (gt % CPR), vr0 = gt >> 2, vc0 = 8 * (gt & 3);
  const int ldv = static_cast<int>(p.ldv);
  auto fetch = [&](__amdgpu_buffer_rsrc_t r, int lane_off, int uniform_off) {
    return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(r, 4 * lane_off, 4 * uniform_off, 0));
  };
  // (no branch around the loads: where two paths of a prefetch join, the
  // compiler waits for it)
  auto load_k = [&](int j0) {  // rows past the keys: the last one
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int off = min(j0 + i * (256 / CPR) + kr0, p.kn - 1) * D + kc0;
      ld[i][0] = fetch(rK, off, 0);
      ld[i][1] = fetch(rK, off + 4, 0);
    }
  };
  auto load_v = [&](int j0) {  // keys past the row: its last four
    const int a = vr0 * ldv + min(j0 + vc0, ldv - 4), b = vr0 * ldv + min(j0 + vc0 + 4, ldv - 4);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      ld[i][0] = fetch(rV, a, i * 64 * ldv);
      ld[i][1] = fetch(rV, b, i * 64 * ldv);
    }
  };
  // chunk c of key row r at c ^ swizzle: the 16 rows of a fragment read
  // (r / 4 % 2 fixed) hit distinct banks
  auto kswizzle = [](int r) { return D >= 128 ? (r & 3) | ((r >> 1) & 12) : ((r >> 1) & 1) | ((r >> 2) & 6); };
  auto store = [&](__bf16* dst, const bf16x8* pl) {
#pragma unroll
    for (int s = 0; s < 3; ++s) *reinterpret_cast<bf16x8*>(dst + s * kPlane) = pl[s];
  };
  auto put_k = [&](int j0) {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int ci = i * 256 + gt, r = ci / CPR, c = ci % CPR;
      bf16x8 pl[3];
      split8(ld[i][0], ld[i][1], pl[0], pl[1], pl[2]);
      m = largest(m, ld[i][0], ld[i][1]);
      store(planes + r * D + ((c ^ kswizzle(r)) << 3), pl);
    }
    if (__builtin_expect(__ballot(m >= kLarge) != 0, 0)) {
      int key = kNone;
#pragma unroll
      for (int i = CH - 1; i >= 0; --i)
        if (largest(0, ld[i][0], ld[i][1]) >= kLarge) key = j0 + (i * 256 + gt) / CPR;
      first_large = min(first_large, wave_least(key));
    }
  };
  auto put_v = [&](int j0) {
    uint32_t m = 0xffffffffu;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int ci = i * 256 + gt, r = ci >> 2, c = ci & 3, key = j0 + 8 * c;
      float4_t a = ld[i][0], b = ld[i][1];
      if (key + 8 > p.kn) {  // keys past kn may be uninitialised
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (key + e >= p.kn) a[e] = 0.0f;
          if (key + 4 + e >= p.kn) b[e] = 0.0f;
        }
      }
      m = least(m, a, b);
      bf16x8 pl[3];
      split8(a, b, pl[0], pl[1], pl[2]);
      store(planes + r * 32 + ((c ^ ((r >> 2) & 3)) << 3), pl);
    }
    if (__builtin_expect(__ballot(m < kTiny - 1u) != 0, 0)) {
      int first = kNone;
#pragma unroll
      for (int e = 7; e >= 0; --e) {
        const int key = j0 + vc0 + e;
        bool tiny = false;
#pragma unroll
        for (int i = 0; i < CH; ++i) tiny |= 2u * __float_as_uint(ld[i][e >> 2][e & 3]) - 1u < kTiny - 1u;
        if (tiny && key < p.kn) first = key;
      }
      first_tiny = min(first_tiny, wave_least(first));
    }
  };

  float4_t O[NDT];
#pragma unroll
  for (int t = 0; t < NDT; ++t) O[t] = float4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.0f, alpha = 1.0f;
  bf16x8 pf[3];
  const int key_end = min(p.kn, offset + q0 + BQ);  // exclusive causal limit of the last row
  const int ntiles = (key_end + BK - 1) / BK, steps = (ntiles + 1) / 2;
  const int lim = min(offset + q0 + 16 * wq + n, p.kn - 1);  // the query's last visible key
  auto row_max = [](float x) {
    x = fmaxf(x, __shfl_xor(x, 16, 64));
    return fmaxf(x, __shfl_xor(x, 32, 64));
  };
  constexpr int PD = 3;  // fragment sets in registers
  const int krow = (8 * (n >> 2) + (n & 3)) * D, kkey = kswizzle(8 * (n >> 2) + (n & 3));  // tile 1: 4 rows on, same key
  auto scores = [&](int j0) {
    // step i: key tile i % 2, k-step i / 2; fragments of two steps in flight
    float4_t hi[2], lo[2];
    hi[0] = hi[1] = lo[0] = lo[1] = float4_t{0.f, 0.f, 0.f, 0.f};
    bf16x8 kf[PD][3], ql[2][2];
    auto read = [&](int i) {
      const int t = i & 1, kb = i >> 1;
#pragma unroll
      for (int s = 0; s < 3; ++s)
        kf[i % PD][s] = *reinterpret_cast<const bf16x8*>(
            planes + krow + s * kPlane + 4 * t * D + (((4 * (kb & 3) + g) ^ kkey) << 3) + (kb >> 2) * 128);
      if (t == 0) {
        ql[kb & 1][0] = qml[kb * 128];
        ql[kb & 1][1] = qml[kb * 128 + 64];
      }
    };
#pragma unroll
    for (int i = 0; i < PD - 1; ++i) read(i);
#pragma unroll
    for (int i = 0; i < 2 * NKB; ++i) {
      if (i + PD - 1 < 2 * NKB) read(i + PD - 1);
      __builtin_amdgcn_sched_barrier(0);
      const int t = i & 1, kb = i >> 1;
      const bf16x8* k3 = kf[i % PD];
#pragma unroll
      for (int q = 0; q < 5; ++q)
        lo[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            k3[kPA[q]], kPB[q] == 0 ? qf[kb] : ql[kb & 1][kPB[q] - 1 < 0 ? 0 : kPB[q] - 1], lo[t], 0, 0, 0);
      hi[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k3[0], qf[kb], hi[t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    // lane (n, g): keys j0 + 8 g + 4 t + i of query n
    float s[8], mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = (hi[t][i] + lo[t][i]) * p.scale;
        s[4 * t + i] = j0 + 8 * g + 4 * t + i > lim ? -INFINITY : v;
        mx = fmaxf(mx, s[4 * t + i]);
      }
    const float mn = fmaxf(m, row_max(mx));
    alpha = m == -INFINITY ? 0.0f : expf(m - mn);
    m = mn;
    float4_t pa, pb;
    float rs = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float pv = s[e] == -INFINITY ? 0.0f : expf(s[e] - mn);
      rs += pv;
      if (e < 4)
        pa[e] = pv;
      else
        pb[e - 4] = pv;
    }
    rs += __shfl_xor(rs, 16, 64);
    rs += __shfl_xor(rs, 32, 64);
    l = l * alpha + rs;
    split8(pa, pb, pf[0], pf[1], pf[2]);
  };
  auto values = [&] {
    const __bf16* vr = planes + n * 32 + ((g ^ ((n >> 2) & 3)) << 3);
    bf16x8 vf[PD][3];
    auto read = [&](int t) {
#pragma unroll
      for (int s = 0; s < 3; ++s) vf[t % PD][s] = *reinterpret_cast<const bf16x8*>(vr + s * kPlane + t * 512);
    };
#pragma unroll
    for (int t = 0; t < PD - 1; ++t) read(t);
    float4_t last = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NDT; ++t) {
      if (t + PD - 1 < NDT) read(t + PD - 1);
      __builtin_amdgcn_sched_barrier(0);
      float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < 6; ++q)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[t % PD][kPA[q]], pf[kPB[q]], acc, 0, 0, 0);
      if (t > 0)  // under the next tile's products
#pragma unroll
        for (int i = 0; i < 4; ++i) O[t - 1][i] = fmaf(O[t - 1][i], alpha, last[i]);
      last = acc;
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) O[NDT - 1][i] = fmaf(O[NDT - 1][i], alpha, last[i]);
  };

  // the phases of a tile: K to LDS | scores | V to LDS | values; group 1 runs
  // one phase behind, so one group splits while the other multiplies
  const int first = grp * BK;
  if (first < key_end) load_k(first);
  if (grp == 1) lds_barrier();
  for (int st = 0; st < steps; ++st) {
    const int j0 = first + st * 2 * BK;
    const bool here = j0 < key_end;
    if (here) {
      put_k(j0);
      load_v(j0);
    }
    lds_barrier();
    if (here) scores(j0);
    lds_barrier();
    if (here) {
      put_v(j0);
      if (j0 + 2 * BK < key_end) load_k(j0 + 2 * BK);
    }
    lds_barrier();
    if (here) values();
    lds_barrier();
  }
  if (grp == 0) lds_barrier();

  // group 1 hands (m, l, O) over; group 0 combines and stores
  float* const mo = reinterpret_cast<float*>(smem) + (wq * 64 + lane) * 4;
  float* const ml = reinterpret_cast<float*>(smem) + 4 * 64 * NDT * 4 + (wq * 64 + lane) * 2;
  if (grp == 1) {
#pragma unroll
    for (int t = 0; t < NDT; ++t) *reinterpret_cast<float4_t*>(mo + t * (4 * 64 * 4)) = O[t];
    ml[0] = m;
    ml[1] = l;
  }
  if (tid < 2) flags[tid] = kNone;
  const int row = q0 + 16 * wq + n, rowc = min(row, p.qn - 1);
  float4_t gv[NDT];  // requested here: behind the barriers they are in
  if (grp == 0) {
    const float* gate = static_cast<const float*>(p.gate) + (int64_t)rowc * p.ldg + (int64_t)h * p.hsg + 4 * g;
#pragma unroll
    for (int t = 0; t < NDT; ++t) {
      if (p.vec_io) {
        gv[t] = *reinterpret_cast<const float4_t*>(gate + 16 * t);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) gv[t][i] = gate[16 * t + i];
      }
    }
  }
  lds_barrier();
  if (lane == 0) {
    if (first_large != kNone) atomicMin(&flags[0], first_large);
    if (first_tiny != kNone) atomicMin(&flags[1], first_tiny);
  }
  lds_barrier();
  if (grp == 0) {
    const float m1 = ml[0], mn = fmaxf(m, m1);
    const float a0 = expf(m - mn), a1 = m1 == -INFINITY ? 0.0f : expf(m1 - mn);  // (key 0 is in group 0: m is not -inf)
    const float inv = 1.0f / (l * a0 + ml[1] * a1);
    const bool tiny = flags[1] <= lim;
    bool odd = flags[0] <= lim || (large_q >> lane & 1) != 0;
#pragma unroll
    for (int t = 0; t < NDT; ++t) {
      const float4_t o1 = *reinterpret_cast<const float4_t*>(mo + t * (4 * 64 * 4));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = (O[t][i] * a0 + o1[i] * a1) * inv;
        odd |= !(fabsf(a) < INFINITY) || (tiny && fabsf(a) < kSmallOut);
        O[t][i] = a;
      }
    }
    // a query's outputs are spread over four lanes
    uint64_t rows = __ballot(odd);
    rows |= rows >> 32;
    rows = (rows | rows >> 16) & 0xffff;
    if (lane == 0) flags[2 + wq] = static_cast<int>(rows);
    float* y = static_cast<float*>(p.y) + (int64_t)rowc * p.ldy + (int64_t)h * D + 4 * g;
    // (rows to form again are not stored here: a caller may gate in place)
    const bool here = row < p.qn && !(rows >> n & 1);
#pragma unroll
    for (int t = 0; t < NDT; ++t) {
      float4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = O[t][i] * (1.0f / (1.0f + expf(-gv[t][i])));
      if (!here) continue;
      if (p.vec_io) {
        *reinterpret_cast<float4_t*>(y + 16 * t) = o;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) y[16 * t + i] = o[i];
      }
    }
  }
  lds_barrier();
  uint64_t again = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w)
    again |= (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(flags[2 + w]) << (16 * w);
  if (again == 0) return;
  lds_barrier();  // the flags' place is attn_body's from here on
  attn_body<float, D, 512>(p, smem, again);
}

// d of a whole tile, 16-byte aligned rows, a head's keys and values within 31-bit byte offsets
inline bool attn_f32_split_ok(const AttnParams& p) {
  return (p.d == 64 || p.d == 128 || p.d == 256) && p.ldv % 4 == 0 && (int64_t)p.kn * p.d < (int64_t(1) << 29) &&
         (int64_t)p.ldv * p.d < (int64_t(1) << 29) &&
         ((reinterpret_cast<uintptr_t>(p.q) | reinterpret_cast<uintptr_t>(p.k) | reinterpret_cast<uintptr_t>(p.vt)) & 15) == 0;
}

inline int attn_f32_split_launch(const AttnParams& p0, hipStream_t s) {
  AttnParams p = p0;
  p.vec_io = ((reinterpret_cast<uintptr_t>(p.gate) | reinterpret_cast<uintptr_t>(p.y)) & 15) == 0 && p.ldg % 4 == 0 &&
             p.hsg % 4 == 0 && p.ldy % 4 == 0;
  const dim3 grid(((p.qn + 63) / 64) * p.heads);
  if (p.d == 64)
    hipLaunchKernelGGL((attn_f32_split<64>), grid, dim3(512), 0, s, p);
  else if (p.d == 128)
    hipLaunchKernelGGL((attn_f32_split<128>), grid, dim3(512), 0, s, p);
  else
    hipLaunchKernelGGL((attn_f32_split<256>), grid, dim3(512), 0, s, p);
  return check_launch("attention");
}
