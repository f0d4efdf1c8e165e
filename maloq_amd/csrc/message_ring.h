#pragma once
// The SO(2) GEMM of the fused message block in bf16: the plans, epilogues and
// outputs of message_gemm.h, bit for bit.
//
// What bounds it: at one wave per 32 x 32 product block every weight fragment
// (1 KB) feeds one MFMA (32 cycles) per row tile, and the four SIMDs of a compute
// unit together draw their operands at the rate of the LDS.  36 800 edges, mmax = lmax
// = 4, 128 channels, first convolution: with the weights read from L2 by each wave, one
// wave per SIMD, 1190 us; so 843 (MFMA 18 % busy, L2 hits 89 %: what is left is the
// latency of a phase, with one workgroup per compute unit).
//   * A workgroup owns NG groups of RT row tiles and CB = 32 kernel-output
//     channels.  Four waves per group own whole output degrees (the schedule of
//     GPlan); the groups share the weights, which are read once per workgroup.
//   * The K loop runs over (l_in, 16 channels).  A phase is KSUB(l_in) steps: all
//     row and weight fragments of the degree, about the same bytes for each
//     degree, copied global -> LDS by DMA into a ring of NST stages, NST - 1 phases
//     ahead, with one barrier per phase.
//   * Within a step a wave reads each operand row once per order and each weight
//     fragment of its degrees once.
#include "message_split.h"

namespace maloq {
namespace msg {

template <int L, int M, bool GATE, int RT, int NG, int MODE>
struct RingGemm {
  using G = Gemm<L, M, GATE, 4, RT, BF16, MODE>;
  using P = typename G::P;
  using S = SplitGemm<L, M, GATE, RT, NG, 1, MODE>;  // kinds and packed positions
  static constexpr int TE = P::TE, NWT = 4 * NG, NR = RT * NG;
  static constexpr bool GOUT = S::GOUT;
  static_assert(NWT % NR == 0, "a wave stages rows of one row tile");

  // ------------------------------------------------------------ stages
  // Of degree li per K step: nA row fragments ([row type][row tile]) and nB weight
  // fragments (in packed order); a stage holds the row fragments of all its steps,
  // then the weight fragments.
  static constexpr int nA(int li) { return P::nqa(li) * NR; }
  static constexpr int nB(int li) { return P::nbfrag(li); }
  static constexpr int CAP = nA(L) + nB(L);  // fragments of a stage
  static constexpr int ksub(int li) {
    const int k = CAP / (nA(li) + nB(li));
    return k >= 4 ? 4 : (k >= 2 ? 2 : 1);
  }
  static constexpr int frags(int li) { return ksub(li) * (nA(li) + nB(li)); }
  static constexpr int slots(int li) { return (frags(li) + NWT - 1) / NWT; }
  static constexpr int NS = [] {
    int m = 1;
    for (int li = 0; li <= L; ++li) m = slots(li) > m ? slots(li) : m;
    return m;
  }();
  static constexpr int NSMIN = [] {
    int m = NS;
    for (int li = 0; li <= L; ++li) m = slots(li) < m ? slots(li) : m;
    return m;
  }();
  static constexpr int STAGE = CAP * FRAG;
  static constexpr int NST = 3 * STAGE + NG * static_cast<int>(sizeof(typename G::Smem)) <= 163840 ? 3 : 2;

  // What slot k of wave w copies for degree li: -1 nothing, else a row of an edge or
  // WEIGHT | packed position, and its step of the phase; then the degree's steps,
  // packed fragments per step and fragments per stage.  A wave keeps its entries in
  // lanes of a few registers (v_readlane).
  static constexpr int WEIGHT = 1 << 30, STEP = 16;
  static constexpr int PER_LI = NS + 3;
  static constexpr int TREGS = ((L + 1) * PER_LI + 63) / 64;
  struct Tab {
    int v[NWT][TREGS * 64];
  };
  static constexpr Tab make_tab() {
    Tab t{};
    for (int w = 0; w < NWT; ++w)
      for (int li = 0; li <= L; ++li) {
        int* e = t.v[w] + li * PER_LI;
        const int A = nA(li) * ksub(li), F = frags(li);
        for (int k = 0; k < NS; ++k) {
          // (past the end: the last weight fragment once more, so that every wave
          // has the same number of copies in flight)
          const int f = w + NWT * k < F ? w + NWT * k : F - 1;
          if (k >= slots(li))
            e[k] = -1;
          else if (f < A)
            e[k] = f / nA(li) << STEP | P::arow(f % nA(li) / NR, li);
          else
            e[k] = WEIGHT | (f - A) / nB(li) << STEP | (f - A) % nB(li);
        }
        e[NS] = ksub(li);
        e[NS + 1] = nB(li);
        e[NS + 2] = F;
      }
    return t;
  }
  static constexpr Tab tab = make_tab();

  static constexpr int POOL = [] {
    int m = NST * STAGE;
    if (MODE != FWD_EDGE && MODE != BWD_EDGE && NWT * G::PW > m) m = NWT * G::PW;
    if (NG * S::GXB > m) m = NG * S::GXB;
    return m;
  }();

  struct Ctx {
    const char* arow;   // this lane's edge's rows (its staging row tile), + 8 h channels
    const char* wp;     // packed weights of the channel block, + this lane's place in a fragment
    int64_t row;        // bytes of a row
    int nks, wave;
    unsigned pool;      // LDS address of the stages
    int tab[TREGS];
  };
  // The next phase to be copied: where its slots' bytes are (advanced from phase to
  // phase; looked up only when the degree changes or its last steps are fewer).
  struct Cursor {
    int li, ks, stage;
    int ksub, nbf;           // of degree li
    int64_t foff;            // packed fragments before degree li's
    bool more;
    uint64_t at[NS];         // this lane's address
    unsigned step[NS];       // bytes from one phase to the next
    unsigned dst[NS];        // in a stage
  };
  static __device__ __forceinline__ int entry(const Ctx& c, int i) {
    int v = __builtin_amdgcn_readlane(c.tab[0], i & 63);
#pragma unroll
    for (int r = 1; r < TREGS; ++r)
      if (i >> 6 == r) v = __builtin_amdgcn_readlane(c.tab[r], i & 63);
    return v;
  }
  static __device__ __forceinline__ void aim(Cursor& n, const Ctx& c) {
    const int e0 = n.li * PER_LI, F = entry(c, e0 + NS + 2);
    n.ksub = entry(c, e0 + NS);
    n.nbf = entry(c, e0 + NS + 1);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const int what = entry(c, e0 + k);
      const bool w = (what & WEIGHT) != 0;
      int s = n.ks + ((what & ~WEIGHT) >> STEP);  // past the last step: that one's, not read
      s = s < c.nks ? s : c.nks - 1;
      const int at = what & ((1 << STEP) - 1), f = c.wave + NWT * k < F ? c.wave + NWT * k : F - 1;
      n.at[k] = what < 0 ? 0
                         : reinterpret_cast<uint64_t>(w ? c.wp : c.arow) +
                               (w ? (n.foff + static_cast<int64_t>(s) * n.nbf + at) * FRAG : at * c.row + s * 32);
      n.step[k] = n.ksub * (w ? n.nbf * FRAG : 32);
      n.dst[k] = what < 0 ? ~0u : f * FRAG;
    }
  }
  static __device__ __forceinline__ void copy(Cursor& n, const Ctx& c) {
    if (!n.more) return;
    const unsigned base = c.pool + n.stage * STAGE;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      if (k >= NSMIN && n.dst[k] == ~0u) continue;
      asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(n.at[k]),
                   "s"(__builtin_amdgcn_readfirstlane(base + n.dst[k]))
                   : "memory", "m0");
    }
    n.stage = n.stage + 1 == NST ? 0 : n.stage + 1;
    n.ks += n.ksub;
    if (n.ks + n.ksub <= c.nks) {
#pragma unroll
      for (int k = 0; k < NS; ++k) n.at[k] += n.step[k];
      return;
    }
    if (n.ks >= c.nks) {
      n.ks = 0;
      n.foff += static_cast<int64_t>(c.nks) * n.nbf;
      if (++n.li > L) {
        n.more = false;
        return;
      }
    }
    aim(n, c);
  }

  // ------------------------------------------------------------ products
  static __device__ __forceinline__ frag_t frag(const char* at) { return *reinterpret_cast<const frag_t*>(at); }
  template <int q>
  static __device__ __forceinline__ void read_a(frag_t (&x)[RT], const char* A, int grp) {
#pragma unroll
    for (int r = 0; r < RT; ++r) x[r] = frag(A + (q * NR + grp * RT + r) * FRAG);
  }
  template <int s0, int stride>
  static __device__ __forceinline__ void mul(f32x16 (&acc)[P::MSLOT], const frag_t (&x)[RT], const frag_t& w) {
    static_for<RT>([&](auto R) {
      constexpr int r = decltype(R)::value;
      mfma(acc[s0 + r * stride], x[r], w, BF16{});
    });
  }
  // One K step of degree LI: row fragments at A, weights at B (+ this lane's 16 bytes).
  template <int W, int LI>
  static __device__ __forceinline__ void step(f32x16 (&acc)[P::MSLOT], const char* A, const char* B, int grp) {
    static_for<S::nkinds(LI)>([&](auto T) {
      constexpr int kind = S::kind_at(LI, decltype(T)::value);
      if constexpr (kind == 0 || kind > M) {
        frag_t x[RT];
        read_a<kind == 0 ? 0 : P::nq(LI)>(x, A, grp);
        static_for<L + 1>([&](auto LO) {
          constexpr int lo = decltype(LO)::value;
          if constexpr (P::tab.owner[lo] == W) {
            constexpr int sb = P::tab.base[lo], st = P::ntype(lo);
            mul<sb, st>(acc, x, frag(B + S::bpos(LI, kind, lo) * FRAG));
            if constexpr (kind == 0 && GOUT && P::gacc(lo)) mul<sb + 1, st>(acc, x, frag(B + S::bpos(LI, 0, L + lo) * FRAG));
          }
          if constexpr (kind == 0 && P::gown(W, lo))
            mul<P::tab.gbase[lo], 1>(acc, x, frag(B + S::bpos(LI, 0, L + lo) * FRAG));
        });
      } else {
        constexpr int m = kind;
        frag_t xp[RT], xm[RT];
        constexpr bool any = [] {
          for (int lo = m; lo <= L; ++lo)
            if (P::tab.owner[lo] == W) return true;
          return false;
        }();
        if constexpr (any) {
          read_a<2 * m - 1>(xp, A, grp);
          read_a<2 * m>(xm, A, grp);
        }
        static_for<L + 1>([&](auto LO) {
          constexpr int lo = decltype(LO)::value;
          if constexpr (P::tab.owner[lo] == W && lo >= m) {
            constexpr int sb = P::tab.base[lo], st = P::ntype(lo);
            constexpr int sp = sb + P::qtype(2 * m - 1, lo), sm = sb + P::qtype(2 * m, lo);
            const frag_t wr = frag(B + S::bpos(LI, m, 2 * (lo - m)) * FRAG);
            const frag_t wi = frag(B + S::bpos(LI, m, 2 * (lo - m) + 1) * FRAG);
            const frag_t wn = neg_frag(wi, BF16{});
            // forward: y+ += Wr x+ - Wi x-, y- += Wi x+ + Wr x-; input gradient:
            // dx+ += Wr dy+ + Wi dy-, dx- += -Wi dy+ + Wr dy-.  Each sum in the
            // order of Gemm::mma_m, for the same bits.
            if constexpr (!P::BWD) {
              mul<sm, st>(acc, xp, wi);
              mul<sp, st>(acc, xp, wr);
              mul<sm, st>(acc, xm, wr);
              mul<sp, st>(acc, xm, wn);
            } else {
              mul<sp, st>(acc, xp, wr);
              mul<sm, st>(acc, xm, wr);
              mul<sp, st>(acc, xm, wi);
              mul<sm, st>(acc, xp, wn);
            }
          }
        });
      }
    });
  }

  template <int W, bool RAD>
  static __device__ __forceinline__ void body(typename G::Smem& s, char* pool, const Args& a, const Ctx& c, Cursor& n,
                                              int cb, int grp, int lane, int nvalid) {
    f32x16 acc[P::MSLOT];
#pragma unroll
    for (int k = 0; k < P::MSLOT; ++k)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[k][i] = 0.f;
    int cur = 0;
    static_for<L + 1>([&](auto LIc) {
      constexpr int LI = decltype(LIc)::value;
      for (int ks = 0; ks < c.nks; ks += ksub(LI)) {
        // this wave's copies of the phase are done (the next phase's may be in
        // flight); after the barrier all waves' are, and the stage read a phase ago
        // is free
        if (NST == 3 && n.more)
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NSMIN) : "memory");
        else
          asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        copy(n, c);
        const int steps = c.nks - ks < ksub(LI) ? c.nks - ks : ksub(LI);
        const char* A = pool + cur * STAGE + lane * 16;
        const char* B = A + nA(LI) * ksub(LI) * FRAG;
        for (int t = 0; t < steps; ++t, A += nA(LI) * FRAG, B += nB(LI) * FRAG) step<W, LI>(acc, A, B, grp);
        cur = cur + 1 == NST ? 0 : cur + 1;
      }
    });
    __syncthreads();  // the stages are the epilogue's staging now
    char* gbase = pool + grp * S::GXB;
    G::template epilogue<W, RAD>(acc, s, a, cb, lane, nvalid, reinterpret_cast<float*>(pool + (4 * grp + W) * G::PW),
                                 gbase, gbase + S::GXB / 3, gbase + 2 * (S::GXB / 3));
  }

  template <bool RAD>
  static __device__ __forceinline__ void run(const Args& a) {
    __shared__ typename G::Smem s[NG];
    __shared__ alignas(16) char pool[POOL];
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
    const int64_t tile = wt * NG + grp, e0 = tile * TE;
    const int nvalid = e0 < a.E ? static_cast<int>((a.E - e0) < TE ? (a.E - e0) : TE) : 0;
    G::setup(s[grp], a, tile, e0, nvalid, tid - 256 * grp, safe);
    Ctx c;
    {
      const int64_t e = wt * NG * TE + wave % NR * 32 + (lane & 31);
      const int64_t ei = e < a.E ? (a.eidx ? a.eidx[e] : e) : safe;
      c.arow = static_cast<const char*>(a.a_src) + (ei * P::DPA * a.C_k + 8 * (lane >> 5)) * 2;
      c.wp = a.wpack + static_cast<int64_t>(cb) * a.frags_per_cb * FRAG + weight_lane(lane);
      c.row = static_cast<int64_t>(a.C_k) * 2;
      c.nks = a.C_k / BF16::KC;
      c.wave = wave;
      c.pool = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) char*)pool));
#pragma unroll
      for (int r = 0; r < TREGS; ++r) c.tab[r] = tab.v[wave][64 * r + lane];
    }
    Cursor n{};
    n.more = true;
    aim(n, c);
    __syncthreads();
    for (int i = 0; i < NST - 1; ++i) copy(n, c);
    // waves w and w + 4 share a SIMD: the second group's run the schedule backwards,
    // so that a heavy wave shares its SIMD with a light one
    const int sw = (wave & 3) ^ (grp & 1 ? 3 : 0);
    static_for<4>([&](auto WI) {
      constexpr int w = decltype(WI)::value;
      if (sw == w) body<w, RAD>(s[grp], pool, a, c, n, cb, grp, lane, nvalid);
    });
  }
};

template <int L, int M, bool GATE, int RT, int NG, int MODE, bool RAD>
__global__ __launch_bounds__(256 * NG, 1) void ring_gemm_kernel(Args a) {
  RingGemm<L, M, GATE, RT, NG, MODE>::template run<RAD>(a);
}

}  // namespace msg
}  // namespace maloq
