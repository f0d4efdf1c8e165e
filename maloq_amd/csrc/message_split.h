#pragma once
// The SO(2) GEMM of the fused message block in fp32, on the bf16 matrix cores
// (split_bf16.h): the same products, epilogues and outputs as message_gemm.h.
//
// What bounds it: six bf16 MFMAs stand for one fp32 product block, so a K step
// of 16 channels is long (4800 cycles per CU at lmax 4, mmax 2) and the loads
// are easily hidden; what competes with the MFMAs is the splitting of the operands on
// the VALU and the LDS reads (no bank conflicts).  36 800 edges, lmax 4, mmax 2, 128
// channels: forward 1296 us on the fp32 matrix instructions, so 957 (942 TFLOP/s of
// bf16 products, where a large library product reaches 1157); input gradient 1432
// and 1209 (727: its epilogue with radial rows spills 200 bytes per lane).  Both ask
// for as much reuse of a split fragment as the registers allow:
//   * A workgroup owns NG tiles of 32 RT edges and CB = 32 kernel-output
//     channels.  Four waves per tile own whole output degrees (the schedule of
//     GPlan); the NG groups share the weights.
//   * The K loop runs over (l_in, 16 channels, kind): kind 0 holds the m = 0
//     rows (and the forward's gate outputs), kind m the +-m rows, kind mmax + 1
//     the gate-gradient rows of the gated input gradient.  A kind's fragments
//     (32 rows x 16 channels, rows and weights alike) are loaded as fp32, split
//     once per workgroup and kept as three planes of 1 KB in LDS; 16 KB x 3 at
//     lmax 4, twice: while one kind is computed the next, loaded a kind earlier,
//     is split and written (one barrier per kind).  A wave stages fragments w,
//     w + 4 NG, ...
//   * Within a kind a wave holds one operand row's planes and one (Wr, Wi) pair
//     at a time beside its accumulators.
//   * Where the tiles leave compute units idle, two groups of waves (KS = 2) halve
//     one tile's K steps between them, each with stages of its own, so that one
//     computes while the other waits; the second's sums are added to the first's.
//   * A tile with a sum that is not finite runs its K loop once more, for infinite
//     operands (split_bf16.h).
#include "message_gemm.h"
#include "split_bf16.h"

namespace maloq {
namespace msg {

template <int L, int M, bool GATE, int RT, int NG, int KS, int MODE>
struct SplitGemm {
  static_assert(NG == 1 || KS == 1, "groups share either the weights or the tile");
  using G = Gemm<L, M, GATE, 4, RT, F32, MODE>;
  using P = typename G::P;
  static constexpr int TE = P::TE;
  static constexpr int NWT = 4 * NG;  // waves that stage one kind
  static constexpr int NR = RT * NG;  // row tiles
  static constexpr int SF = 3 * FRAG;  // bytes of a split fragment
  static constexpr bool GOUT = GATE && !P::BWD, GIN = GATE && P::BWD;
  static constexpr int d = (L + 1) * (L + 1);
  static_assert(NWT % NR == 0, "a wave stages rows of one row tile");

  // ------------------------------------------------------------ kinds
  static constexpr int KINDS = M + 1 + (GIN ? 1 : 0);
  static constexpr bool has(int li, int kind) { return kind <= M ? kind <= li : li >= 1; }
  // the kinds of degree li in order
  static constexpr int nkinds(int li) { return cmin(M, li) + 1 + (GIN && li >= 1 ? 1 : 0); }
  static constexpr int kind_at(int li, int t) { return t <= cmin(M, li) ? t : M + 1; }
  static constexpr int nA(int kind) { return (kind >= 1 && kind <= M ? 2 : 1) * NR; }
  static constexpr int nB(int kind) {
    return kind == 0 ? L + 1 + (GOUT ? L : 0) : (kind <= M ? 2 * (L + 1 - kind) : L + 1);
  }
  static constexpr int slots(int kind) { return (nA(kind) + nB(kind) + NWT - 1) / NWT; }
  static constexpr int NS = [] {
    int m = 1;
    for (int k = 0; k < KINDS; ++k) m = slots(k) > m ? slots(k) : m;
    return m;
  }();
  static constexpr int STAGE = [] {
    int m = 0;
    for (int k = 0; k < KINDS; ++k) m = nA(k) + nB(k) > m ? nA(k) + nB(k) : m;
    return m * SF;
  }();
  // packed position, among the fragments of (li, K step), of weight fragment j of a kind
  static constexpr int bpos(int li, int kind, int j) {
    if (kind == 0) return j <= L ? P::bbase(li, j) : P::bbase(li, j - L) + 1;
    if (kind > M) return P::bbase(li, j) + 1;
    const int lo = kind + j / 2;
    return P::bbase(li, lo) + 1 + P::gt(lo) + P::gin(li) + 2 * (kind - 1) + j % 2;
  }
  // row (within an edge's rows) of operand row qi of a kind
  static constexpr int arow(int li, int kind, int qi) {
    return kind == 0 ? P::arow(0, li) : (kind <= M ? P::arow(2 * kind - 1 + qi, li) : P::arow(P::nq(li), li));
  }

  // What slot k of wave w stages for the t-th kind of degree li: -1 nothing, an
  // operand row, or WEIGHT | packed position; and each degree's number of kinds
  // and of packed fragments per 8 channels.  A wave keeps its own entries in
  // lanes of a few registers (v_readlane: a scalar load would wait for the LDS
  // reads in flight).
  static constexpr int WEIGHT = 1 << 30;
  static constexpr int PER_LI = KINDS * NS + 2;
  static constexpr int ENTRIES = (L + 1) * PER_LI;
  static constexpr int TREGS = (ENTRIES + 63) / 64;
  struct StageTab {
    int v[NWT][TREGS * 64];
  };
  static constexpr StageTab make_stages() {
    StageTab t{};
    for (int w = 0; w < NWT; ++w)
      for (int li = 0; li <= L; ++li) {
        int* e = t.v[w] + li * PER_LI;
        for (int i = 0; i < nkinds(li); ++i) {
          const int kind = kind_at(li, i);
          for (int k = 0; k < NS; ++k) {
            const int f = w + NWT * k;
            e[i * NS + k] = f < nA(kind) ? arow(li, kind, f / NR)
                                         : (f < nA(kind) + nB(kind) ? WEIGHT | bpos(li, kind, f - nA(kind)) : -1);
          }
        }
        e[KINDS * NS] = nkinds(li);
        e[KINDS * NS + 1] = P::nbfrag(li);
      }
    return t;
  }
  static constexpr StageTab stages = make_stages();

  // ------------------------------------------------------------ LDS
  // After the K loop the stages hold the epilogue's per-wave staging, and before
  // it (gate rows apart) the gate values of each group.
  static constexpr int GXB = P::GW ? 3 * G::GPS * RT * 16 * 64 * 4 : 0;  // per group
  static constexpr int POOL = [] {
    int m = KS * 2 * STAGE;
    if (MODE != FWD_EDGE && MODE != BWD_EDGE && KS * NWT * G::PW > m) m = KS * NWT * G::PW;
    if (KS * NG * GXB > m) m = KS * NG * GXB;
    return m;
  }();

  struct Ctx {
    const char* arow;   // this lane's edge's rows (its staging row tile), + 4 h
    const char* wp;     // packed weights of the channel block, + this lane's place in a fragment
    int C_k;
    int nks8;           // 8-channel blocks
    int ks0, nks;       // first of this group's K steps per degree, and their number
    int wave;           // among those that stage together
    int tab[TREGS];     // entry 64 r + lane of this wave's staging table
  };

  // ------------------------------------------------------------ staging
  // Fragments on their way to LDS: the next kind's, loaded a whole kind before
  // they are needed (rows come from HBM).
  struct Flight {
    frag_t v[NS][2];
    int what[NS];            // as in the table
    int valid;               // 8-channel blocks of the step: 2, 1 or none
    int li, ks, t;           // of the fragments in v
    int nk, nbf;             // of degree li
    int foff;                // packed fragments before degree li's
    bool more;               // a kind is left
    int again;               // sums formed again, for infinite operands (split_bf16.h)
  };
  static __device__ __forceinline__ int entry(const Ctx& c, int i) {
    int v = __builtin_amdgcn_readlane(c.tab[0], i & 63);
#pragma unroll
    for (int r = 1; r < TREGS; ++r)
      if (i >> 6 == r) v = __builtin_amdgcn_readlane(c.tab[r], i & 63);
    return v;
  }
  // Where this lane's part of the cursor's fragments is: found before the
  // registers of the last ones are free, so that the loads can be issued back to
  // back (an address in a register that a load may still write would have to wait
  // for all of them).
  struct Addr {
    uint64_t p[NS];
    uint32_t step[NS];
    int what[NS];
    int valid;
  };
  static __device__ __forceinline__ void locate(Addr& d, const Flight& n, const Ctx& c) {
    // channels are a multiple of 8: the last step may be half (its second half is
    // read from the first, and zeroed when it is split), and the second of two
    // groups' last one empty
    const int left = c.nks8 - 2 * n.ks, ks = KS > 1 && left <= 0 ? n.ks - 1 : n.ks;
    d.valid = left;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const int what = entry(c, n.li * PER_LI + n.t * NS + k);
      const bool w = (what & WEIGHT) != 0;
      const uint32_t off = w ? static_cast<uint32_t>(n.foff + 2 * ks * n.nbf + (what ^ WEIGHT)) * FRAG
                             : static_cast<uint32_t>(what * c.C_k + 16 * ks) * 4;
      d.what[k] = what;
      d.step[k] = 2 * ks + 1 >= c.nks8 ? 0 : (w ? static_cast<uint32_t>(n.nbf) * FRAG : 32);
      const uint64_t base = w ? reinterpret_cast<uint64_t>(c.wp) : reinterpret_cast<uint64_t>(c.arow);
      uint64_t at = base + off;
      asm volatile("" : "+v"(at));
      d.p[k] = at;
    }
  }
  static __device__ __forceinline__ void load(Flight& n, const Addr& d) {
    n.valid = d.valid;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      n.what[k] = d.what[k];
      if (d.what[k] < 0) continue;
      typedef const __attribute__((address_space(1))) frag_t* global_frag;
      n.v[k][0] = *reinterpret_cast<global_frag>(d.p[k]);
      n.v[k][1] = *reinterpret_cast<global_frag>(d.p[k] + d.step[k]);
    }
  }
  static __device__ __forceinline__ void store(const Flight& n, const Ctx& c, char* buf, int lane) {
    char* at = buf + c.wave * SF + lane * 16;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      if (n.what[k] < 0) continue;
      float r[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r[i] = KS > 1 && n.valid < 1 ? 0.f : __uint_as_float(n.v[k][0][i]);
        r[4 + i] = n.valid < 2 ? 0.f : __uint_as_float(n.v[k][1][i]);
      }
      uint4 pl[3];
      split8(r, pl);
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4*>(at + NWT * k * SF + i * FRAG) = pl[i];
    }
    if (__builtin_expect(n.again, 0)) {
      int held = 0;
#pragma unroll
      for (int k = 0; k < NS; ++k) held |= (n.what[k] >= 0) << k;
#pragma unroll 1
      for (int k = 0; k < NS; ++k)
        if (held >> k & 1) fix_inf(at + NWT * k * SF, FRAG);
    }
  }
  static __device__ __forceinline__ void degree(Flight& n, const Ctx& c, int li) {
    n.li = li;
    n.nk = entry(c, li * PER_LI + KINDS * NS);
    n.nbf = entry(c, li * PER_LI + KINDS * NS + 1);
  }
  static __device__ __forceinline__ void advance(Flight& n, const Ctx& c) {
    if (++n.t < n.nk) return;
    n.t = 0;
    if (++n.ks < c.ks0 + c.nks) return;
    n.ks = c.ks0;
    n.foff += c.nks8 * n.nbf;
    if (n.li == L)
      n.more = false;
    else
      degree(n, c, n.li + 1);
  }

  // ------------------------------------------------------------ products
  struct Frag3 {
    frag_t p[3];
  };
  static __device__ __forceinline__ void read3(Frag3& x, const char* at) {
#pragma unroll
    for (int i = 0; i < 3; ++i) x.p[i] = *reinterpret_cast<const frag_t*>(at + i * FRAG);
  }
  template <int kind, int qi>
  static __device__ __forceinline__ void read_a(Frag3 (&x)[RT], const char* buf, int grp) {
    static_for<RT>([&](auto R) {
      constexpr int r = decltype(R)::value;
      read3(x[r], buf + (qi * NR + r) * SF + grp * (RT * SF));
    });
  }
  // acc[slot(r)] += weight x row tile r, for two (weight, accumulator) pairs
  template <int s0, int s1, int stride>
  static __device__ __forceinline__ void mul2(f32x16 (&acc)[P::MSLOT], const Frag3 (&x)[RT], const Frag3& w0,
                                              const Frag3& w1) {
#pragma unroll
    for (int k = 0; k < SPLIT_PRODUCTS; ++k)
      static_for<RT>([&](auto R) {
        constexpr int r = decltype(R)::value;
        mfma(acc[s0 + r * stride], x[r].p[split_a(k)], w0.p[split_b(k)], BF16{});
        mfma(acc[s1 + r * stride], x[r].p[split_a(k)], w1.p[split_b(k)], BF16{});
      });
  }
  template <int s0, int stride>
  static __device__ __forceinline__ void mul1(f32x16 (&acc)[P::MSLOT], const Frag3 (&x)[RT], const Frag3& w0) {
#pragma unroll
    for (int k = 0; k < SPLIT_PRODUCTS; ++k)
      static_for<RT>([&](auto R) {
        constexpr int r = decltype(R)::value;
        mfma(acc[s0 + r * stride], x[r].p[split_a(k)], w0.p[split_b(k)], BF16{});
      });
  }
  // One kind of one K step, from stage `buf` (+ this lane's 16 bytes); `mid` runs
  // between its two halves.
  template <int W, int LI, int kind, class F>
  static __device__ __forceinline__ void compute(f32x16 (&acc)[P::MSLOT], const char* buf, int grp, F&& mid) {
    constexpr int B0 = nA(kind);
    if constexpr (kind == 0 || kind > M) {
      Frag3 x[RT];
      read_a<kind, 0>(x, buf, grp);
      static_for<L + 1>([&](auto LO) {
        constexpr int lo = decltype(LO)::value;
        if constexpr (P::tab.owner[lo] == W) {
          constexpr int sb = P::tab.base[lo];
          Frag3 w;
          read3(w, buf + (B0 + lo) * SF);
          mul1<sb, P::ntype(lo)>(acc, x, w);
          if constexpr (kind == 0 && GOUT && P::gacc(lo)) {
            read3(w, buf + (B0 + L + lo) * SF);
            mul1<sb + 1, P::ntype(lo)>(acc, x, w);
          }
        }
        if constexpr (kind == 0 && P::gown(W, lo)) {
          Frag3 w;
          read3(w, buf + (B0 + L + lo) * SF);
          mul1<P::tab.gbase[lo], 1>(acc, x, w);
        }
      });
      mid();
    } else {
      constexpr int m = kind;
      constexpr int last = [] {  // the wave's last degree with order m
        int k = -1;
        for (int lo = m; lo <= L; ++lo)
          if (P::tab.owner[lo] == W) k = lo;
        return k;
      }();
      if constexpr (last < 0) mid();
      static_for<L + 1>([&](auto LO) {
        constexpr int lo = decltype(LO)::value;
        if constexpr (P::tab.owner[lo] == W && lo >= m) {
          constexpr int sb = P::tab.base[lo], st = P::ntype(lo);
          constexpr int sp = sb + P::qtype(2 * m - 1, lo), sm = sb + P::qtype(2 * m, lo);
          Frag3 wr, wi, x[RT];
          read3(wr, buf + (B0 + 2 * (lo - m)) * SF);
          read3(wi, buf + (B0 + 2 * (lo - m) + 1) * SF);
          // forward: y+ += Wr x+ - Wi x-, y- += Wi x+ + Wr x-; input gradient:
          // dx+ += Wr dy+ + Wi dy-, dx- += -Wi dy+ + Wr dy-.  The half with +Wi
          // first, then Wi is negated in place.
          if constexpr (!P::BWD) {
            read_a<kind, 0>(x, buf, grp);
            mul2<sp, sm, st>(acc, x, wr, wi);
          } else {
            read_a<kind, 1>(x, buf, grp);
            mul2<sm, sp, st>(acc, x, wr, wi);
          }
          if constexpr (lo == last) mid();
#pragma unroll
          for (int i = 0; i < 3; ++i) wi.p[i] = neg_frag(wi.p[i], BF16{});
          if constexpr (!P::BWD) {
            read_a<kind, 1>(x, buf, grp);
            mul2<sm, sp, st>(acc, x, wr, wi);
          } else {
            read_a<kind, 0>(x, buf, grp);
            mul2<sp, sm, st>(acc, x, wr, wi);
          }
        }
      });
    }
  }

  static __device__ __forceinline__ void barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's LDS writes are done
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }

  // One kind of one K step of degree LI from the stage at `cur`; between its
  // halves the next kind's fragments go to the other stage and the loads of the
  // one after it are issued.  At entry every wave has written its part of this
  // stage and left the other one (the barrier that ended the last kind).
  template <int W, int LI, int kind>
  static __device__ __forceinline__ void phase(f32x16 (&acc)[P::MSLOT], const Ctx& c, Flight& n, char* pool, int& cur,
                                               int grp, int lane) {
    compute<W, LI, kind>(acc, pool + cur + lane * 16, grp, [&] {
      if (n.more) {
        const Flight now = n;
        Addr at;
        advance(n, c);
        locate(at, n, c);  // past the end: the last kind's, not loaded
        store(now, c, pool + (STAGE - cur), lane);
        if (n.more) load(n, at);
      }
    });
    barrier();
    cur = STAGE - cur;
  }

  // The first kind into the stage at 0, the second's loads issued.
  static __device__ __forceinline__ void begin(Flight& n, const Ctx& c, char* stages, int lane) {
    n.more = true;
    n.ks = c.ks0;
    n.t = n.foff = 0;
    degree(n, c, 0);
    Addr at;
    locate(at, n, c);
    load(n, at);
    store(n, c, stages, lane);
    advance(n, c);
    locate(at, n, c);
    if (n.more) load(n, at);
    __syncthreads();
  }

  template <int W, bool RAD>
  static __device__ __forceinline__ void body(typename G::Smem& s, int* again, char* pool, const Args& a, const Ctx& c,
                                              Flight& n, int cb, int grp, int lane, int nvalid) {
    char* stages = pool + (KS > 1 ? grp * 2 * STAGE : 0);
    f32x16 acc[P::MSLOT];
#pragma unroll 1
    for (n.again = 0;;) {
      begin(n, c, stages, lane);
#pragma unroll
      for (int k = 0; k < P::MSLOT; ++k)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[k][i] = 0.f;
      int cur = 0;
      static_for<L + 1>([&](auto LIc) {
        constexpr int LI = decltype(LIc)::value;
        for (int ks = 0; ks < c.nks; ++ks)
          static_for<nkinds(LI)>([&](auto T) {
            phase<W, LI, kind_at(LI, decltype(T)::value)>(acc, c, n, stages, cur, KS > 1 ? 0 : grp, lane);
          });
      });
      if (n.again) break;
      float t[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < P::MSLOT; ++k)
#pragma unroll
        for (int i = 0; i < 16; ++i) t[i & 3] = not_finite(t[i & 3], acc[k][i]);
      t[0] = (t[0] + t[1]) + (t[2] + t[3]);
      if (t[0] != t[0]) *again = 1;
      __syncthreads();
      // (every wave's; the asm keeps two copies of the loop from being made of it)
      n.again = __builtin_amdgcn_readfirstlane(*again);
      asm volatile("" : "+s"(n.again));
      if (__builtin_expect(!n.again, 1)) break;
    }
    // every wave is past its last read of the stages: they are staging now
    if constexpr (KS > 1) {
      constexpr int CH = POOL / (4 * FRAG * 4);  // accumulators at a time
      static_assert(CH > 0, "no room for the second group's sums");
      static_for<(P::MSLOT + CH - 1) / CH>([&](auto I) {
        constexpr int k0 = decltype(I)::value * CH, k1 = k0 + CH < P::MSLOT ? k0 + CH : P::MSLOT;
        auto at = [&](int k, int i) {
          return reinterpret_cast<f32x4*>(pool + ((W * CH + k - k0) * 4 + i) * FRAG + lane * 16);
        };
        if (grp == 1) {
#pragma unroll
          for (int k = k0; k < k1; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              *at(k, i) = f32x4{acc[k][4 * i], acc[k][4 * i + 1], acc[k][4 * i + 2], acc[k][4 * i + 3]};
        }
        __syncthreads();
        if (grp == 0) {
#pragma unroll
          for (int k = k0; k < k1; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const f32x4 v = *at(k, i);
#pragma unroll
              for (int j = 0; j < 4; ++j) acc[k][4 * i + j] += v[j];
            }
        }
        __syncthreads();
      });
    }
    char* gbase = pool + grp * GXB;
    G::template epilogue<W, RAD>(acc, s, a, cb, lane, nvalid,
                                 reinterpret_cast<float*>(pool + (4 * grp + W) * G::PW), gbase, gbase + GXB / 3,
                                 gbase + 2 * (GXB / 3));
  }

  template <bool RAD>
  static __device__ __forceinline__ void run(const Args& a) {
    __shared__ typename G::Smem s[NG * KS];
    __shared__ alignas(16) char pool[POOL];
    __shared__ int again;  // a sum is not finite
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // XCD-aware mapping, as in Gemm::run, over groups of NG tiles
    const int64_t bid = blockIdx.x;
    const int64_t slot = bid >> 3;
    const int cb = a.cb0 + static_cast<int>(slot % a.n_cb);
    const int64_t wt = (slot / a.n_cb) * 8 + (bid & 7);
    if (wt * NG >= a.ntiles) return;  // whole workgroup exits together
    const int safe = a.eidx ? a.eidx[wt * NG * TE] : static_cast<int>(wt * NG * TE);
    const int grp = wave >> 2;
    // (the second group of two on one tile: a tile without edges, for the epilogue)
    const int64_t tile = KS > 1 && grp > 0 ? a.ntiles : wt * NG + grp;
    const int64_t e0 = tile * TE;
    const int nvalid = e0 < a.E ? static_cast<int>((a.E - e0) < TE ? (a.E - e0) : TE) : 0;
    G::setup(s[grp], a, tile, e0, nvalid, tid - 256 * grp, safe);
    if (tid == 0) again = 0;
    Ctx c;
    {
      const int rt = wave % NR;  // staging row tile
      const int64_t e = wt * NG * TE + rt * 32 + (lane & 31);
      const int64_t ei = e < a.E ? (a.eidx ? a.eidx[e] : e) : safe;
      c.arow = static_cast<const char*>(a.a_src) + (ei * P::DPA * a.C_k + 4 * (lane >> 5)) * 4;
      c.wp = a.wpack + static_cast<int64_t>(cb) * a.frags_per_cb * FRAG + weight_lane(lane);
      c.C_k = a.C_k;
      c.nks8 = a.C_k / 8;
      c.nks = ((c.nks8 + 1) / 2 + KS - 1) / KS;
      c.ks0 = KS > 1 ? grp * c.nks : 0;
      c.wave = KS > 1 ? wave & 3 : wave;
#pragma unroll
      for (int r = 0; r < TREGS; ++r) c.tab[r] = stages.v[c.wave][64 * r + lane];
    }
    Flight n{};
    // waves w and w + 4 share a SIMD: the second group's run the schedule backwards,
    // so that a heavy wave shares its SIMD with a light one
    const int sw = (wave & 3) ^ (grp & 1 ? 3 : 0);
    static_for<4>([&](auto WI) {
      constexpr int w = decltype(WI)::value;
      if (sw == w) body<w, RAD>(s[grp], &again, pool, a, c, n, cb, grp, lane, nvalid);
    });
  }
};

template <int L, int M, bool GATE, int RT, int NG, int KS, int MODE, bool RAD>
__global__ __launch_bounds__(256 * NG * KS, 1) void split_gemm_kernel(Args a) {
  SplitGemm<L, M, GATE, RT, NG, KS, MODE>::template run<RAD>(a);
}

}  // namespace msg
}  // namespace maloq
