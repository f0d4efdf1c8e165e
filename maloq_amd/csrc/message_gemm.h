#pragma once
// The SO(2) GEMM of the fused message block with its inverse-rotation and
// sorted-segment-sum epilogue (gfx950, MFMA 32x32).
//
// Input rows: Y [E, d', C_k] (m-major kept rows of D x[src] (*) rad, written by
// the prep kernel) for the forward; the rotated output gradient for the input
// gradient (edges in source order, rows gathered through eidx).
//
// Work split.  A workgroup (NW waves) owns TE = 32 RT consecutive edges of the
// segment-sorted order and CB = 32 kernel-output channels.  Each wave owns a
// set of whole output degrees l_out (compile-time longest-processing-time
// schedule over the MFMA work of each degree) for all RT row tiles, so the
// inverse rotation runs from its own accumulators and the segment sum stays
// inside the wave.  The K loop runs over (l_in, KC input channels):
//   * A (rotated rows): one 1 KB fragment per (row type q of l_in, row tile),
//     in the exact lane order of the MFMA A operand, copied global -> LDS by
//     DMA (global_load_lds) into a ring of three stages, two steps ahead; one
//     barrier per step.  Every wave reads the fragments it needs from LDS.
//   * B (weights): each wave loads only the fragments of its own degrees
//     straight from global memory into registers (16 bytes per lane, fully
//     coalesced; packed on the host in lane order), one step ahead.  For
//     m > 0 only Wr and Wi are stored; the complex mix
//         y+ = Wr x+ - Wi x-,  y- = Wi x+ + Wr x-        (so2_layers.py:61-67)
//     and its transpose (input gradient: dx+ = Wr^T dy+ + Wi^T dy-,
//     dx- = -Wi^T dy+ + Wr^T dy-) negate a register copy of Wi.
// The weights are the MFMA's A operand and the rows its B operand, so an
// accumulator lane holds one edge (lane & 31) and 16 consecutive channels of
// the block (half h = lane >> 5: channels 16 h + i in register i; the weight
// fragment's lanes are read through a permutation that makes them consecutive).
// Everything that is per edge in the epilogue is then per lane: its kept Wigner
// entries, its saved rows, radial scales and gate rows are 16-byte loads and
// stores of the lane's own edge, with no transposition through LDS.  (With lane =
// channel those went through LDS, edge by edge: 45 000 edges, lmax 6, 128 channels,
// bf16, gated 1105 us forward and 1087 input gradient, so 1023 and 1038.)
// Epilogue per owned degree l: [bias, gate | radial scale and its gradient],
// then for each pair of output columns (j, j+1) and each 32-edge row tile:
// v = sum_q D(q, j) acc_q in the lane, written to a per-wave LDS tile
// [edge][2 columns x 32 channels] and read back with lane = (column, channel);
// the sum over the edges runs in order with uniform control (segment ends from
// a 64-bit ballot mask); each finished segment is stored once (or to the
// partials buffer when it is cut by a tile boundary).  Deterministic: fixed
// summation order, no atomics.
#include "message_impl.h"

namespace maloq {
namespace msg {

// MODE FWD: a gated block has one more output row type per degree l >= 1 (the
// gate pre-activations); MODE BWD_DX: one more input row type per degree
// l >= 1 (dL/dgate), whose products with the transposed gate weights add to
// the m = 0 outputs.
template <int L, int M, bool GATE, int NW, int RT, int MODE = 0>
struct GPlan {
  static constexpr int TE = 32 * RT;
  static constexpr int NT = NW * 64;
  static_assert(TE <= 64, "segment masks are 64-bit");
  static constexpr bool BWD = MODE == 1 || MODE == 3;  // BWD_DX, BWD_EDGE
  static constexpr int gt(int l) { return (GATE && !BWD && l >= 1) ? 1 : 0; }   // output gate row
  static constexpr int gin(int l) { return (GATE && BWD && l >= 1) ? 1 : 0; }   // input gate row
  static constexpr int nq(int l) { return 1 + 2 * cmin(M, l); }
  static constexpr int nqa(int l) { return nq(l) + gin(l); }  // A row types of input degree l
  // Gate rows apart (GW): a gated forward at lmax 6, mmax < lmax puts the gate
  // row of each degree l >= 1 in the wave with the fewest accumulators at that
  // point (the wave left without a degree, then those of the light degrees),
  // so the waves of the heavy degrees hold only their kept rows; the gate
  // values reach a degree's wave through LDS after the K loop.
  static constexpr bool GW = GATE && !BWD && L > 4 && M < L;
  static constexpr int gacc(int l) { return GW ? 0 : gt(l); }  // gate row among degree l's accumulators
  static constexpr int ntype(int l) { return nq(l) + gacc(l); }
  // accumulator type of row type q of degree l (0: m=0, [1: gate], then +1, -1, +2, ...)
  static constexpr int qtype(int q, int l) { return q == 0 ? 0 : q + gacc(l); }
  static constexpr int DP = Plan<L, M, false, 4, 1>::DP;
  static constexpr int DPA = DP + ((GATE && BWD) ? L : 0);  // A rows per edge
  // A-source row of input row type q of degree l (gate rows follow the kept rows)
  static constexpr int arow(int q, int l) { return q < nq(l) ? Plan<L, M, false, 4, 1>::mrow(q, l) : DP + l - 1; }
  static constexpr int mrow(int q, int l) { return Plan<L, M, false, 4, 1>::mrow(q, l); }
  static constexpr int doff(int l) { return Plan<L, M, false, 4, 1>::doff(l); }
  static constexpr int DS = Plan<L, M, false, 4, 1>::DS;
  // B fragments of one K step (kernel-input degree li), grouped by output degree lo:
  // g0, [gate], then (Wr, Wi) for m = 1 .. min(M, li, lo).
  static constexpr int nbl(int li, int lo) { return 1 + gt(lo) + gin(li) + 2 * cmin(cmin(M, li), lo); }
  static constexpr int bbase(int li, int lo) {
    int s = 0;
    for (int k = 0; k < lo; ++k) s += nbl(li, k);
    return s;
  }
  static constexpr int nbfrag(int li) { return bbase(li, L + 1); }
  // B registers of degree lo at li in its own wave (with GW the gate fragment
  // is the gate wave's), and the packed position of that wave's fragment t
  static constexpr int nblr(int li, int lo) { return nbl(li, lo) - gt(lo) + gacc(lo); }
  static constexpr int bpos(int lo, int t) { return t == 0 ? 0 : t + gt(lo) - gacc(lo); }
  // MFMAs per row tile and K step summed over li: the schedule's weight of degree lo
  static constexpr int work(int lo) {
    int s = 0;
    for (int li = 0; li <= L; ++li) s += 1 + gacc(lo) + gin(li) + 4 * cmin(cmin(M, li), lo);
    return s;
  }
  struct Tab {
    int owner[L + 1];
    int base[L + 1];   // first accumulator slot of degree l in its wave
    int nslots[NW];
    int gowner[L + 1];  // GW: wave holding the gate row of degree l >= 1
    int gbase[L + 1];   // GW: its accumulator slots gbase .. gbase + RT - 1 (one per row tile)
  };
  static constexpr Tab make() {
    Tab t{};
    int load[NW] = {};
    bool done[L + 1] = {};
    for (int it = 0; it <= L; ++it) {
      int best = -1;
      for (int l = L; l >= 0; --l)
        if (!done[l] && (best < 0 || work(l) > work(best))) best = l;
      int w = 0;
      for (int k = 1; k < NW; ++k)
        if (load[k] < load[w]) w = k;
      t.owner[best] = w;
      load[w] += work(best);
      done[best] = true;
    }
    for (int w = 0; w < NW; ++w) {
      int s = 0;
      for (int l = 0; l <= L; ++l)
        if (t.owner[l] == w) {
          t.base[l] = s;
          s += RT * ntype(l);
        }
      t.nslots[w] = s;
    }
    if (GW)
      for (int l = 1; l <= L; ++l) {
        int w = 0;
        for (int k = 1; k < NW; ++k)
          if (t.nslots[k] < t.nslots[w]) w = k;
        t.gowner[l] = w;
        t.gbase[l] = t.nslots[w];
        t.nslots[w] += RT;
      }
    return t;
  }
  static constexpr Tab tab = make();
  static constexpr bool gown(int w, int l) { return GW && l >= 1 && tab.gowner[l] == w; }
  static constexpr bool has_deg(int w) {
    for (int l = 0; l <= L; ++l)
      if (tab.owner[l] == w) return true;
    return false;
  }
  // B registers of wave w at li: degree lo's fragments start at wboff(w, li, lo),
  // then (GW) the gate fragment of each gate row it holds, at gboff(w, li, lo)
  static constexpr int wboff(int w, int li, int lo) {
    int s = 0;
    for (int k = 0; k < lo; ++k)
      if (tab.owner[k] == w) s += nblr(li, k);
    return s;
  }
  static constexpr int gboff(int w, int li, int lo) {
    int s = wboff(w, li, L + 1);
    for (int k = 1; k < lo; ++k)
      if (gown(w, k)) ++s;
    return s;
  }
  static constexpr int nbw(int w, int li) { return gboff(w, li, L + 1); }
  static constexpr int NBW = [] {
    int m = 1;
    for (int w = 0; w < NW; ++w) m = nbw(w, L) > m ? nbw(w, L) : m;
    return m;
  }();
  static constexpr int MSLOT = [] {
    int m = 1;
    for (int w = 0; w < NW; ++w) m = tab.nslots[w] > m ? tab.nslots[w] : m;
    return m;
  }();
  // Wigner rows: the pair-major layout of the dk workspace
  static constexpr int pblk(int l) { return PairLayout<L, M>::pblk(l); }
  static constexpr int woff(int l) { return PairLayout<L, M>::woff(l); }
  static constexpr int WS = PairLayout<L, M>::WS;
  // LDS
  static constexpr int A_BYTES = nqa(L) * RT * FRAG;     // one A stage
  static constexpr int NA = (nqa(L) * RT * 64 + NT - 1) / NT;  // A chunks per thread
};

// One lane's 16 bytes of an MFMA operand fragment (a native vector, so that
// arrays of fragments are promoted to registers).
typedef unsigned int frag_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ frag_t neg_frag(frag_t v, BF16) { return v ^ 0x80008000u; }
__device__ __forceinline__ frag_t neg_frag(frag_t v, F32) { return v ^ 0x80000000u; }
// acc += (weight fragment w)^T (row fragment a): accumulator rows are output
// channels, columns (lanes) edges.
__device__ __forceinline__ void mfma(f32x16& acc, frag_t a, frag_t w, BF16) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16((bf16x8)w, (bf16x8)a, acc, 0, 0, 0);
}
// Lane half h holds channels 4 h .. 4 h + 3 of an 8-wide K step: instruction j pairs
// channels j and 4 + j of both operands.
__device__ __forceinline__ void mfma(f32x16& acc, frag_t a, frag_t w, F32) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(w[j]), __uint_as_float(a[j]), acc, 0, 0, 0);
}

// Byte offset in a packed weight fragment (lane i: column i & 31) that lane
// `lane` reads: accumulator row r = 8 a + 4 h + b then holds channel 16 h + 4 a + b,
// so register 4 a + b of a lane of half h is channel 16 h + 4 a + b.
__device__ __forceinline__ int weight_lane(int lane) {
  const int r = lane & 31;
  return ((lane & 32) + 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3)) * 16;
}

template <int L, int M, bool GATE, int NW, int RT, class TM, int MODE>
struct Gemm {
  using P = GPlan<L, M, GATE, NW, RT, MODE>;
  static constexpr int TE = P::TE, NT = P::NT, KC = TM::KC;
  static constexpr int d = (L + 1) * (L + 1);

  struct Smem {
    float* optr[TE];  // destination row block of the segment ending at each edge
    int seg[TE];
    int eid[TE];  // -1 past the tile's edges
    int safe;     // an edge id that may be read in their place
  };
  // A stages (three distinct LDS objects, so the compiler can tell a stage
  // being filled by DMA from the one being read); after the K loop they hold
  // the epilogue's per-wave staging, WPS waves per stage (2 of 4 waves: st0
  // and st1; 3 of 8 waves: all three): 32 edges x 64 floats, padded to 68 (16-byte
  // rows; the writes of 8 lanes and the reads of a row are free of bank conflicts).
  static constexpr int TP = 68;
  static constexpr int PW = 32 * TP * 4;
  static constexpr int WPS = (NW + 2) / 3;
  // Gate wave (P::GW): after the K loop the stages also carry tanh of the gate
  // rows to the degree waves, degree l's RT x 16 x 64 floats in stage (l - 1) / GPS.
  static constexpr int GPS = (L + 2) / 3;
  static constexpr int GXB = P::GW ? GPS * RT * 16 * 64 * 4 : 0;
  static constexpr int SB0 = (P::A_BYTES > WPS * PW) ? P::A_BYTES : WPS * PW;
  static constexpr int SB = SB0 > GXB ? SB0 : GXB;
  static __device__ __forceinline__ float* wave_staging(int wave, char* st0, char* st1, char* st2) {
    const int k = wave / WPS;
    return reinterpret_cast<float*>((k == 0 ? st0 : (k == 1 ? st1 : st2)) + (wave - k * WPS) * PW);
  }
  typedef __attribute__((address_space(3))) void lds_void;

  // ------------------------------------------------------------ A operand
  // A staging: the nq(L) RT fragments of a K step are split over the waves,
  // waves with the least MFMA work taking the most (their registers are free);
  // wave W stages the fragments f with stager(f) == W, k-th of them in slot k.
  // Row type q = f / RT, row tile f % RT; lane (row, half) copies 16 bytes of
  // its edge's row.  Which fragments exist is a compile-time property of
  // (W, k, LI), so every load is unconditional (which keeps the compiler's
  // vmcnt accounting exact); lanes of edges beyond the tile read the tile's
  // first edge, whose rows in those accumulator lanes are never stored.
  struct ATab {
    int frag[NW][P::nqa(L) * RT];
    int count[NW];
  };
  static constexpr ATab make_atab() {
    ATab t{};
    int order[NW] = {};
    for (int w = 0; w < NW; ++w) order[w] = w;
    for (int i = 0; i < NW; ++i)  // waves by ascending MFMA slots
      for (int j = i + 1; j < NW; ++j)
        if (P::tab.nslots[order[j]] < P::tab.nslots[order[i]]) {
          const int x = order[i];
          order[i] = order[j];
          order[j] = x;
        }
    constexpr int F = P::nqa(L) * RT;
    for (int f = 0; f < F; ++f) {
      int best = order[0];  // fewest staged so far, ties to the lighter wave
      for (int i = 1; i < NW; ++i) {
        const int w = order[i];
        const int cb = t.count[best] - (best == order[0] ? (F + NW - 1) / NW - F / NW : 0);
        const int cw = t.count[w] - (w == order[0] ? (F + NW - 1) / NW - F / NW : 0);
        if (cw < cb) best = w;
      }
      t.frag[best][t.count[best]++] = f;
    }
    return t;
  }
  static constexpr ATab atab = make_atab();
  static constexpr int NAW = [] {
    int m = 1;
    for (int w = 0; w < NW; ++w) m = atab.count[w] > m ? atab.count[w] : m;
    return m;
  }();
  template <int W, int k>
  static constexpr int afrag() { return atab.frag[W][k]; }
  template <int W, int k, int LI>
  static constexpr bool avalid() { return k < atab.count[W] && afrag<W, k>() < P::nqa(LI) * RT; }

  struct AState {
    int64_t ebase[NAW];  // element offset of (edge, row 0, channel half)
  };

  template <int W>
  static __device__ __forceinline__ void a_init(AState& st, const Smem& s, const Args& a, int lane) {
    static_for<NAW>([&](auto K) {
      constexpr int k = decltype(K)::value;
      if constexpr (k >= atab.count[W]) return;
      constexpr int rt = afrag<W, k>() % RT;
      const int e = rt * 32 + (lane & 31);
      const int ei = s.eid[e] >= 0 ? s.eid[e] : s.safe;
      st.ebase[k] = static_cast<int64_t>(ei) * P::DPA * a.C_k + (lane >> 5) * TM::VEC;
    });
  }
  // Direct global -> LDS copies of this wave's fragments of step (LI, ks):
  // lane i's 16 bytes land at stage + f*FRAG + 16 i, the MFMA lane order.
  template <int W, int LI>
  static __device__ __forceinline__ void a_dma(const AState& st, char* stage, const Args& a, int ks) {
    const typename TM::raw* y = reinterpret_cast<const typename TM::raw*>(a.a_src);
    static_for<NAW>([&](auto K) {
      constexpr int k = decltype(K)::value;
      if constexpr (avalid<W, k, LI>()) {
        constexpr int q = afrag<W, k>() / RT;
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass does not know gfx950's 16-byte form
        __builtin_amdgcn_global_load_lds(
            y + st.ebase[k] + static_cast<int64_t>(P::arow(q, LI)) * a.C_k + ks * KC,
            (lds_void*)(stage + afrag<W, k>() * FRAG), 16, 0, 0);
#endif
      }
    });
  }

  // ------------------------------------------------------------ B operand
  template <int W, int LI>
  static __device__ __forceinline__ void b_load(frag_t (&b)[P::NBW], const char* wp, int64_t foff,
                                                int ks, int lane) {
    const char* base = wp + (foff + static_cast<int64_t>(ks) * P::nbfrag(LI)) * FRAG + weight_lane(lane);
    static_for<L + 1>([&](auto LO) {
      constexpr int lo = decltype(LO)::value;
      if constexpr (P::tab.owner[lo] == W) {
        static_for<P::nblr(LI, lo)>([&](auto T) {
          constexpr int t = decltype(T)::value;
          b[P::wboff(W, LI, lo) + t] =
              *reinterpret_cast<const frag_t*>(base + (P::bbase(LI, lo) + P::bpos(lo, t)) * FRAG);
        });
      }
    });
    static_for<L + 1>([&](auto LO) {  // a gate fragment follows its degree's m = 0 fragment
      constexpr int lo = decltype(LO)::value;
      if constexpr (P::gown(W, lo))
        b[P::gboff(W, LI, lo)] = *reinterpret_cast<const frag_t*>(base + (P::bbase(LI, lo) + 1) * FRAG);
    });
  }

  // ------------------------------------------------------------ MFMA step
  // Fragment (row type q, all row tiles) of the current stage.
  template <int q>
  static __device__ __forceinline__ void read_q(frag_t (&af)[RT], const char* A, int lane) {
    static_for<RT>([&](auto R) {
      constexpr int rt = decltype(R)::value;
      af[rt] = *reinterpret_cast<const frag_t*>(A + (q * RT + rt) * FRAG + lane * 16);
    });
  }
  // m = 0 (and gate) products of every owned degree: forward, the gate
  // outputs from the m = 0 inputs; input gradient, the m = 0 outputs also
  // from the gate-gradient inputs ag.
  template <int W, int LI>
  static __device__ __forceinline__ void mma_m0(f32x16 (&acc)[P::MSLOT], const frag_t (&a0)[RT],
                                                const frag_t (&ag)[RT], const frag_t (&b)[P::NBW]) {
    static_for<L + 1>([&](auto LO) {
      constexpr int lo = decltype(LO)::value;
      if constexpr (P::gown(W, lo))
        static_for<RT>([&](auto R) {
          constexpr int rt = decltype(R)::value;
          mfma(acc[P::tab.gbase[lo] + rt], a0[rt], b[P::gboff(W, LI, lo)], TM{});
        });
    });
    static_for<L + 1>([&](auto LO) {
      constexpr int lo = decltype(LO)::value;
      if constexpr (P::tab.owner[lo] == W) {
        constexpr int bo = P::wboff(W, LI, lo);
        static_for<RT>([&](auto R) {
          constexpr int rt = decltype(R)::value;
          constexpr int sb = P::tab.base[lo] + rt * P::ntype(lo);
          mfma(acc[sb], a0[rt], b[bo], TM{});
          if constexpr (P::gacc(lo)) mfma(acc[sb + 1], a0[rt], b[bo + 1], TM{});
          if constexpr (P::gin(LI)) mfma(acc[sb], ag[rt], b[bo + 1], TM{});
        });
      }
    });
  }
  // +-m products of every owned degree.  Forward: y+ += Wr x+ - Wi x-,
  // y- += Wi x+ + Wr x-; input gradient: dx+ += Wr dy+ + Wi dy-,
  // dx- += -Wi dy+ + Wr dy-.  The negated Wi is formed after the last use of Wi.
  template <int W, int LI, int m>
  static __device__ __forceinline__ void mma_m(f32x16 (&acc)[P::MSLOT], const frag_t (&ap)[RT],
                                               const frag_t (&am)[RT], const frag_t (&b)[P::NBW]) {
    static_for<L + 1>([&](auto LO) {
      constexpr int lo = decltype(LO)::value;
      if constexpr (P::tab.owner[lo] == W && m <= lo) {
        constexpr int bw = P::wboff(W, LI, lo) + 1 + P::gacc(lo) + P::gin(LI) + 2 * (m - 1);
        const frag_t wr = b[bw], wi = b[bw + 1];
        static_for<RT>([&](auto R) {
          constexpr int rt = decltype(R)::value;
          constexpr int sb = P::tab.base[lo] + rt * P::ntype(lo);
          constexpr int sp = sb + P::qtype(2 * m - 1, lo), sm = sb + P::qtype(2 * m, lo);
          if constexpr (!P::BWD) {
            mfma(acc[sm], ap[rt], wi, TM{});
            mfma(acc[sm], am[rt], wr, TM{});
            mfma(acc[sp], ap[rt], wr, TM{});
          } else {
            mfma(acc[sp], ap[rt], wr, TM{});
            mfma(acc[sp], am[rt], wi, TM{});
            mfma(acc[sm], am[rt], wr, TM{});
          }
        });
        const frag_t nwi = neg_frag(wi, TM{});
        static_for<RT>([&](auto R) {
          constexpr int rt = decltype(R)::value;
          constexpr int sb = P::tab.base[lo] + rt * P::ntype(lo);
          if constexpr (!P::BWD)
            mfma(acc[sb + P::qtype(2 * m - 1, lo)], am[rt], nwi, TM{});
          else
            mfma(acc[sb + P::qtype(2 * m, lo)], ap[rt], nwi, TM{});
        });
      }
    });
  }

  // DMA instructions wave W issues for one K step of input degree LI.
  template <int W, int LI>
  static constexpr int ndma() {
    int n = 0;
    for (int k = 0; k < NAW; ++k)
      if (k < atab.count[W] && atab.frag[W][k] < P::nqa(LI) * RT) ++n;
    return n;
  }
  template <int I>
  static __device__ __forceinline__ char* stage(char* s0, char* s1, char* s2) {
    return I == 0 ? s0 : (I == 1 ? s1 : s2);
  }

  // One K step of wave W on input degree LI: A fragments from stage RD, B
  // fragments in bn (loaded by the previous step).  The A stages form a ring of
  // three, filled by DMA two steps ahead; B is loaded one step ahead.  At entry
  // the wave's outstanding vector-memory operations are, in issue order, the B
  // loads of this step and the DMA of the next step (PEND instructions), so
  // vmcnt(PEND) leaves only the latter in flight, and after the barrier every
  // wave's DMA of this step has landed.  lgkmcnt(0): the previous step's LDS
  // reads are complete before any wave refills that stage.  Then: B of the
  // next step (degree NB, K step ksb, fragment base fb; none if NB < 0) into
  // bn, DMA of the step after it (degree NA, K step ksa; none if NA < 0) into
  // stage (RD + 2) % 3, and the MFMAs of this step.
  template <int W, int LI, int RD, int NB, int NA, int PEND>
  static __device__ __forceinline__ void kstep(f32x16 (&acc)[P::MSLOT], frag_t (&bn)[P::NBW],
                                               const AState& st, char* s0, char* s1, char* s2,
                                               const Args& a, const char* wp, int64_t fb, int ksb,
                                               int ksa, int lane) {
    // s_waitcnt as a builtin, so that the compiler's own wait insertion counts it
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((PEND & 15) | (7 << 4) | ((PEND >> 4) << 14));  // vmcnt(PEND) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    frag_t bc[P::NBW];
#pragma unroll
    for (int i = 0; i < P::NBW; ++i) bc[i] = bn[i];
    if constexpr (NB >= 0) b_load<W, NB>(bn, wp, fb, ksb, lane);
    if constexpr (NA >= 0) a_dma<W, NA>(st, stage<(RD + 2) % 3>(s0, s1, s2), a, ksa);
    // keep the next steps' loads ahead of this step's MFMAs
    __builtin_amdgcn_sched_barrier(0);
    const char* rd = stage<RD>(s0, s1, s2);
    frag_t a0[RT], ag[RT];
    read_q<0>(a0, rd, lane);
    if constexpr (P::gin(LI)) read_q<P::nq(LI)>(ag, rd, lane);
    mma_m0<W, LI>(acc, a0, ag, bc);
    static_for<M>([&](auto MI) {
      constexpr int m = decltype(MI)::value + 1;
      if constexpr (m <= LI && P::has_deg(W)) {
        frag_t ap[RT], am[RT];
        read_q<2 * m - 1>(ap, rd, lane);
        read_q<2 * m>(am, rd, lane);
        mma_m<W, LI, m>(acc, ap, am, bc);
      }
    });
  }

  // The nks K steps of input degree LI.  KR = nks % 3 for nks >= 2 (then the
  // stage of the degree's first step is (LI nks) % 3 = (LI KR) % 3), KR = 3 for
  // nks == 1.  Step ks loads B of ks + 1 and DMAs ks + 2, crossing into degree
  // LI + 1 for the last two steps; the ring position of every step is static.
  template <int W, int LI, int KR>
  static __device__ __forceinline__ void kdegree(f32x16 (&acc)[P::MSLOT], frag_t (&bn)[P::NBW],
                                                 const AState& st, char* s0, char* s1, char* s2,
                                                 const Args& a, const char* wp, int64_t foff, int nks,
                                                 int lane) {
    constexpr int NXT = LI < L ? LI + 1 : -1;
    constexpr int ND = ndma<W, LI>();
    if constexpr (KR == 3) {  // one step per degree: B of degree LI + 1, DMA of LI + 2
      constexpr int NA = LI + 2 <= L ? LI + 2 : -1;
      constexpr int PEND = NXT >= 0 ? ndma<W, (NXT >= 0 ? NXT : 0)>() : 0;
      kstep<W, LI, LI % 3, NXT, NA, PEND>(acc, bn, st, s0, s1, s2, a, wp, foff + P::nbfrag(LI), 0, 0, lane);
    } else {
      constexpr int PH = (LI * KR) % 3;
      constexpr int REM = (KR + 1) % 3;  // (nks - 2) % 3
      int ks = 0;
      for (; ks + 3 <= nks - 2; ks += 3) {
        kstep<W, LI, PH, LI, LI, ND>(acc, bn, st, s0, s1, s2, a, wp, foff, ks + 1, ks + 2, lane);
        kstep<W, LI, (PH + 1) % 3, LI, LI, ND>(acc, bn, st, s0, s1, s2, a, wp, foff, ks + 2, ks + 3, lane);
        kstep<W, LI, (PH + 2) % 3, LI, LI, ND>(acc, bn, st, s0, s1, s2, a, wp, foff, ks + 3, ks + 4, lane);
      }
      if constexpr (REM >= 1)
        kstep<W, LI, PH, LI, LI, ND>(acc, bn, st, s0, s1, s2, a, wp, foff, ks + 1, ks + 2, lane);
      if constexpr (REM >= 2)
        kstep<W, LI, (PH + 1) % 3, LI, LI, ND>(acc, bn, st, s0, s1, s2, a, wp, foff, ks + 2, ks + 3, lane);
      constexpr int PEND_NXT = NXT >= 0 ? ndma<W, (NXT >= 0 ? NXT : 0)>() : 0;
      const int64_t fnext = foff + static_cast<int64_t>(nks) * P::nbfrag(LI);
      // ks = nks - 2: B of (LI, nks - 1), DMA of (LI + 1, 0)
      kstep<W, LI, (PH + REM) % 3, LI, NXT, ND>(acc, bn, st, s0, s1, s2, a, wp, foff, nks - 1, 0, lane);
      // ks = nks - 1: B of (LI + 1, 0), DMA of (LI + 1, 1)
      kstep<W, LI, (PH + REM + 1) % 3, NXT, NXT, PEND_NXT>(acc, bn, st, s0, s1, s2, a, wp, fnext, 0, 1,
                                                            lane);
    }
  }

  // ------------------------------------------------------------ epilogue
  // In the accumulators lane (co = lane & 31, h = lane >> 5) holds edge co of the
  // row tile and channels cb CB + 16 h + i, i = 0..15.
  static __device__ __forceinline__ void load16(const typename TM::raw* p, float (&v)[16]) {
    float t[8];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      load_vec<TM, 8>(p + 8 * k, t);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[8 * k + i] = t[i];
    }
  }
  static __device__ __forceinline__ void store16(typename TM::raw* p, const float (&v)[16]) {
    float t[8];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int i = 0; i < 8; ++i) t[i] = v[8 * k + i];
      store_vec<TM, 8>(p + 8 * k, t);
    }
  }
  static __device__ __forceinline__ void store16(typename TM::raw* p, const f32x16& v) {
    float t[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) t[i] = v[i];
    store16(p, t);
  }
  static __device__ __forceinline__ void load_bias(const float* bias, int64_t at, float (&b)[16]) {
    // branch-free: a runtime branch around accumulator updates costs spills
#pragma unroll
    for (int i = 0; i < 16; ++i) b[i] = bias != nullptr ? bias[at + i] : 0.f;
  }

  // col: the lane's first channel
  template <int lo>
  static __device__ __forceinline__ void add_bias(f32x16 (&acc)[P::MSLOT], const Args& a, int col) {
    float b0[16];
    load_bias(a.bias, a.extra + static_cast<int64_t>(lo) * a.C_n + col, b0);
    static_for<RT>([&](auto RTI) {
      constexpr int sb = P::tab.base[lo] + decltype(RTI)::value * P::ntype(lo);
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[sb][i] += b0[i];
    });
    if constexpr (P::gacc(lo)) {
      load_bias(a.bias, static_cast<int64_t>(lo - 1) * a.C_n + col, b0);
      static_for<RT>([&](auto RTI) {
        constexpr int sb = P::tab.base[lo] + decltype(RTI)::value * P::ntype(lo);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[sb + 1][i] += b0[i];
      });
    }
  }

  // Gated forward: the pre-activation rows of degree lo (kept rows and the gate
  // row) to a.gsave [edge id][d' + L][C_n].  ZOUT: the activated kept rows (no
  // gate rows) to a.zout [edge id][d'][C_n] instead (the edge-frame output of
  // FWD_EDGE).
  template <int lo, bool ZOUT = false>
  static __device__ __forceinline__ void save_pre(const f32x16 (&acc)[P::MSLOT], const Smem& s,
                                                  const Args& a, int col, int lane) {
    constexpr int RPE = ZOUT ? P::DP : P::DP + L;  // rows per edge of the destination
    static_for<RT>([&](auto RTI) {
      constexpr int rt = decltype(RTI)::value;
      constexpr int sb = P::tab.base[lo] + rt * P::ntype(lo);
      const int ei = s.eid[rt * 32 + (lane & 31)];
      if (ei < 0) return;
      typename TM::raw* g = reinterpret_cast<typename TM::raw*>(ZOUT ? a.zout : a.gsave) +
                            static_cast<int64_t>(ei) * RPE * a.C_n + col;
      static_for<P::ntype(lo)>([&](auto TI) {
        constexpr int t = decltype(TI)::value;  // accumulator type: 0, [gate], +1, -1, ...
        if constexpr (ZOUT && P::gacc(lo) && t == 1) return;
        constexpr int row = (P::gacc(lo) && t == 1) ? P::DP + lo - 1
                                                    : P::mrow(t == 0 ? 0 : t - P::gacc(lo), lo);
        store16(g + static_cast<int64_t>(row) * a.C_n, acc[sb + t]);
      });
    });
  }

  // ---- gate rows apart (P::GW): wave tab.gowner[l] holds the gate row of
  // degree l, row tile rt, in accumulator tab.gbase[l] + rt.
  // Gate bias, then (with a.gsave) the pre-activation gate rows to a.gsave
  // [edge id][d' + L][C_n], row d' + l - 1.
  template <int W>
  static __device__ __forceinline__ void gate_rows(f32x16 (&acc)[P::MSLOT], const Smem& s, const Args& a,
                                                   int col, int lane) {
    static_for<L + 1>([&](auto LO) {
      constexpr int lo = decltype(LO)::value;
      if constexpr (P::gown(W, lo)) {
        float bg[16];
        load_bias(a.bias, static_cast<int64_t>(lo - 1) * a.C_n + col, bg);
        static_for<RT>([&](auto R) {
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[P::tab.gbase[lo] + decltype(R)::value][i] += bg[i];
        });
      }
    });
    if (a.gsave == nullptr) return;
    static_for<RT>([&](auto RTI) {
      constexpr int rt = decltype(RTI)::value;
      const int ei = s.eid[rt * 32 + (lane & 31)];
      if (ei < 0) return;
      typename TM::raw* gp = reinterpret_cast<typename TM::raw*>(a.gsave) +
                             static_cast<int64_t>(ei) * (P::DP + L) * a.C_n + col;
      static_for<L + 1>([&](auto LO) {
        constexpr int lo = decltype(LO)::value;
        if constexpr (P::gown(W, lo))
          store16(gp + static_cast<int64_t>(P::DP + lo - 1) * a.C_n, acc[P::tab.gbase[lo] + rt]);
      });
    });
  }
  // tanh of the gate row of degree g + 1, row tile rt: register i of lane at
  // gx<g, rt>[i * 64 + lane]
  template <int g, int rt>
  static __device__ __forceinline__ float* gx(char* st0, char* st1, char* st2) {
    constexpr int k = g / GPS;
    return reinterpret_cast<float*>(k == 0 ? st0 : (k == 1 ? st1 : st2)) + ((g % GPS) * RT + rt) * 16 * 64;
  }
  template <int W>
  static __device__ __forceinline__ void gate_out(const f32x16 (&acc)[P::MSLOT], char* st0, char* st1,
                                                  char* st2, int lane) {
    static_for<L + 1>([&](auto LO) {
      constexpr int lo = decltype(LO)::value;
      if constexpr (P::gown(W, lo))
        static_for<RT>([&](auto R) {
          constexpr int rt = decltype(R)::value;
          float* x = gx<lo - 1, rt>(st0, st1, st2);
#pragma unroll
          for (int i = 0; i < 16; ++i) x[i * 64 + lane] = tanhf(acc[P::tab.gbase[lo] + rt][i]);
        });
    });
  }
  // A degree's GateActivation with the gate values from LDS.
  template <int lo>
  static __device__ __forceinline__ void gate_act_gw(f32x16 (&acc)[P::MSLOT], char* st0, char* st1,
                                                     char* st2, int lane) {
    static_for<RT>([&](auto RTI) {
      constexpr int rt = decltype(RTI)::value;
      constexpr int sb = P::tab.base[lo] + rt * P::ntype(lo);
      if constexpr (lo == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float z = acc[sb][i];
          acc[sb][i] = z / (1.0f + __expf(-z));
        }
      } else {
        const float* x = gx<lo - 1, rt>(st0, st1, st2);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float g = x[i * 64 + lane];
          static_for<P::nq(lo)>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            acc[sb + P::qtype(q, lo)][i] *= g;
          });
        }
      }
    });
  }

  // BWD_EDGE with a.gsave: the GateActivation backward (activation.py:57-77)
  // fused into the edge-frame store.  acc holds o = dL/d(gate output) of degree
  // lo; a lane reads the saved pre-activations z of the same edge and channels
  // (and the gate row) and writes to a.zout [edge id][d' + L][C_n]:
  //   lo = 0:  dpre = o s (1 + z (1 - s)),  s = sigmoid(z);
  //   lo >= 1: t = tanh(z_gate); dpre_q = o_q t;  dgate = (1 - t^2) sum_q o_q z_q.
  template <int lo>
  static __device__ __forceinline__ void store_gate_bwd(const f32x16 (&acc)[P::MSLOT], const Smem& s,
                                                        const Args& a, int col, int lane) {
    constexpr int DG = P::DP + L;
    static_for<RT>([&](auto RTI) {
      constexpr int rt = decltype(RTI)::value;
      constexpr int sb = P::tab.base[lo] + rt * P::ntype(lo);
      const int ei = s.eid[rt * 32 + (lane & 31)];
      if (ei < 0) return;
      const int64_t base = static_cast<int64_t>(ei) * DG * a.C_n + col;
      typename TM::raw* g = reinterpret_cast<typename TM::raw*>(a.zout) + base;
      const typename TM::raw* zs = reinterpret_cast<const typename TM::raw*>(a.gsave) + base;
      // Eight channels at a time, the next row's loads under this one's products, each
      // row's offset found where it is used: sixteen channels and kept offsets spilled
      // 320 bytes per lane at mmax = lmax = 4 in bf16 (36 800 edges, 128 channels: 733 us).
      constexpr int VEC = TM::VEC, NU = 8 / VEC;
      auto at = [&](int row, int c0) {
        int64_t o = static_cast<int64_t>(row) * a.C_n + c0;
        asm volatile("" : "+s"(o));
        return o;
      };
      auto fetch = [&](uint4 (&u)[NU], int64_t o) {
#pragma unroll
        for (int k = 0; k < NU; ++k) u[k] = reinterpret_cast<const uint4*>(zs + o)[k];
      };
      auto unpack = [&](const uint4 (&u)[NU], float (&v)[8]) {
#pragma unroll
        for (int k = 0; k < NU; ++k) unpack_vec<TM, VEC>(u[k], *reinterpret_cast<float(*)[VEC]>(&v[k * VEC]));
      };
      static_for<2>([&](auto HI) {
        constexpr int c0 = 8 * decltype(HI)::value;
        float z[8], w[8];
        uint4 u[NU];
        fetch(u, at(P::mrow(0, lo), c0));
        if constexpr (lo == 0) {
          unpack(u, z);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float sg = 1.0f / (1.0f + expf(-z[i]));
            w[i] = acc[sb][c0 + i] * (sg * (1.0f + z[i] * (1.0f - sg)));
          }
          store_vec<TM, 8>(g + at(P::mrow(0, 0), c0), w);
        } else {
          float tg[8], dg[8];
          load_vec<TM, 8>(zs + at(P::DP + lo - 1, c0), tg);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            tg[i] = tanhf(tg[i]);
            dg[i] = 0.f;
          }
          static_for<P::ntype(lo)>([&](auto TI) {
            constexpr int t = decltype(TI)::value;
            unpack(u, z);
            if constexpr (t + 1 < P::ntype(lo)) fetch(u, at(P::mrow(t + 1, lo), c0));
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const float o = acc[sb + t][c0 + i];
              dg[i] = fmaf(o, z[i], dg[i]);
              w[i] = o * tg[i];
            }
            store_vec<TM, 8>(g + at(P::mrow(t, lo), c0), w);
            __builtin_amdgcn_sched_barrier(0);  // one row at a time (register pressure)
          });
#pragma unroll
          for (int i = 0; i < 8; ++i) w[i] = dg[i] * (1.0f - tg[i] * tg[i]);
          store_vec<TM, 8>(g + at(P::DP + lo - 1, c0), w);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  }

  template <int lo>
  static __device__ __forceinline__ void gate_act(f32x16 (&acc)[P::MSLOT]) {
    static_for<RT>([&](auto RTI) {
      constexpr int sb = P::tab.base[lo] + decltype(RTI)::value * P::ntype(lo);
      if constexpr (GATE) {
        if constexpr (lo == 0) {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const float z = acc[sb][i];
            acc[sb][i] = z / (1.0f + __expf(-z));
          }
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const float g = tanhf(acc[sb + 1][i]);
            static_for<P::nq(lo)>([&](auto Q) {
              constexpr int q = decltype(Q)::value;
              acc[sb + P::qtype(q, lo)][i] *= g;
            });
          }
        }
      }
    });
  }

  // Input gradient: the accumulators hold dY (forward-input side) of degree lo.
  // grad_rad = sum_(+-) dY * R (R: unscaled forward rows); dY *= rad.
  template <int lo>
  static __device__ __forceinline__ void radial(f32x16 (&acc)[P::MSLOT], const Smem& s,
                                                const Args& a, int col, int lane) {
    const int64_t rw = rad_width<L, M>(a.C_n);
    static_for<RT>([&](auto RTI) {
      constexpr int rt = decltype(RTI)::value;
      constexpr int sb = P::tab.base[lo] + rt * P::ntype(lo);
      const int ei = s.eid[rt * 32 + (lane & 31)];
      const int64_t eis = ei >= 0 ? ei : s.safe;
      const typename TM::raw* rsave = reinterpret_cast<const typename TM::raw*>(a.rsave) +
                                      eis * P::DP * a.C_n + col;
      // 16-byte pieces at a time: fp32 rows eight channels, bf16 rows all sixteen
      constexpr int NC = sizeof(typename TM::raw) == 2 ? 16 : 8;
      static_for<(1 + (lo < M ? lo : M)) * (16 / NC)>([&](auto MI) {
        constexpr int m = decltype(MI)::value / (16 / NC), c0 = decltype(MI)::value % (16 / NC) * NC;
        constexpr int q0 = m == 0 ? 0 : 2 * m - 1, nqm = m == 0 ? 1 : 2;
        const int64_t slot = rad_slot<L, M>(q0, lo, col, a.C_n) + c0;
        const typename TM::raw* radp = reinterpret_cast<const typename TM::raw*>(a.rad) + eis * rw + slot;
        float rv[NC], dr[NC];
#pragma unroll
        for (int k = 0; k < NC; k += 8) load_vec<TM, 8>(radp + k, *reinterpret_cast<float(*)[8]>(&rv[k]));
#pragma unroll
        for (int i = 0; i < NC; ++i) dr[i] = 0.f;
        static_for<nqm>([&](auto QI) {
          constexpr int q = q0 + decltype(QI)::value;
          constexpr int sl = sb + P::qtype(q, lo);
          float rr[NC];
#pragma unroll
          for (int k = 0; k < NC; k += 8)
            load_vec<TM, 8>(rsave + static_cast<int64_t>(P::mrow(q, lo)) * a.C_n + c0 + k,
                            *reinterpret_cast<float(*)[8]>(&rr[k]));
#pragma unroll
          for (int i = 0; i < NC; ++i) {
            dr[i] = fmaf(acc[sl][c0 + i], rr[i], dr[i]);
            acc[sl][c0 + i] *= rv[i];
          }
        });
        if (a.drad != nullptr && ei >= 0) {
          typename TM::raw* dp = reinterpret_cast<typename TM::raw*>(a.drad) + ei * rw + slot;
#pragma unroll
          for (int k = 0; k < NC; k += 8) store_vec<TM, 8>(dp + k, *reinterpret_cast<float(*)[8]>(&dr[k]));
        }
        __builtin_amdgcn_sched_barrier(0);  // one block at a time (register pressure)
      });
    });
  }

  // Inverse rotation of degree lo and segment sum into out / partials.
  // Per output-column pair p (j = 2p, 2p + 1) and row tile: rotate the lane's
  // edge (its Wigner entries straight from the dk rows, one pair ahead), write
  // both columns to the wave's LDS tile [edge][column][channel], read them back
  // with lane (channel, column) = (lane & 31, lane >> 5), sum over the edges in
  // order, and store the sums of the segments that end in the tile.
  template <int W, int lo>
  static __device__ __forceinline__ void rotate_sum(f32x16 (&acc)[P::MSLOT], Smem& s, const Args& a, int cb,
                                                    float* buf, int lane, uint64_t endmask) {
    constexpr int n = 2 * lo + 1;
    constexpr int nq = P::nq(lo);
    constexpr int PB = P::pblk(lo);
    const int co = lane & 31, h = lane >> 5;
    const int ow = a.ow > 0 ? a.ow : a.C_n;
    const int ocb = a.ow > 0 ? cb - a.cb0 : cb;
    const float4* Dp[RT];
    static_for<RT>([&](auto R) {
      constexpr int rt = decltype(R)::value;
      const int ei = s.eid[rt * 32 + co], e = ei >= 0 ? ei : s.safe;
      Dp[rt] = reinterpret_cast<const float4*>(a.dk + static_cast<int64_t>(e) * P::WS + P::woff(lo));
    });
    float4 nxt[PB / 4];
#pragma unroll
    for (int v = 0; v < PB / 4; ++v) nxt[v] = Dp[0][v];
    float* wr = buf + co * TP + 16 * h;
    const float* rd = buf + lane;
    for (int p = 0; p <= lo; ++p) {
      const bool has_col = 2 * p + h < n;
      const int64_t colo = static_cast<int64_t>(lo * lo + 2 * p + h) * ow + ocb * CB + co;
      float run = 0.f;
      static_for<RT>([&](auto R) {
        constexpr int rt = decltype(R)::value;
        constexpr int sb = P::tab.base[lo] + rt * P::ntype(lo);
        float dv[PB];
#pragma unroll
        for (int v = 0; v < PB / 4; ++v) {
          dv[4 * v] = nxt[v].x; dv[4 * v + 1] = nxt[v].y; dv[4 * v + 2] = nxt[v].z; dv[4 * v + 3] = nxt[v].w;
        }
        {
          const int np = rt + 1 < RT ? p : (p < lo ? p + 1 : lo);
          constexpr int nrt = rt + 1 < RT ? rt + 1 : 0;
#pragma unroll
          for (int v = 0; v < PB / 4; ++v) nxt[v] = Dp[nrt][np * (PB / 4) + v];
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            float o[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              o[k] = 0.f;
              static_for<nq>([&](auto Q) {
                constexpr int q = decltype(Q)::value;
                o[k] = fmaf(dv[2 * q + j], acc[sb + P::qtype(q, lo)][4 * g + k], o[k]);
              });
            }
            *reinterpret_cast<float4*>(wr + 32 * j + 4 * g) = make_float4(o[0], o[1], o[2], o[3]);
          }
        wave_sync();
        // the tile's segment ends, opaque per tile: otherwise the compiler hoists
        // the uniform branches' conditions out of the column loop and spills them
        uint32_t em = static_cast<uint32_t>(endmask >> (32 * rt));
        asm volatile("" : "+s"(em));
        float x[32];
#pragma unroll
        for (int u = 0; u < 32; ++u) x[u] = rd[u * TP];
#pragma unroll
        for (int u = 0; u < 32; u += 4) {
          if (((em >> u) & 15u) == 0u) {
            run += x[u];
            run += x[u + 1];
            run += x[u + 2];
            run += x[u + 3];
          } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              run += x[u + k];
              if ((em >> (u + k)) & 1u) {
                if (has_col) s.optr[rt * 32 + u + k][colo] = run;
                run = 0.f;
              }
            }
          }
        }
        wave_sync();
      });
    }
  }

  // What follows the K loop: the tile's nvalid edges' outputs from the wave's
  // accumulators.  buf: the wave's staging; st0..st2: where the gate values pass
  // from their waves to the degrees' (P::GW).
  template <int W, bool RAD>
  static __device__ __forceinline__ void epilogue(f32x16 (&acc)[P::MSLOT], Smem& s, const Args& a, int cb, int lane,
                                                  int nvalid, float* buf, char* st0, char* st1, char* st2) {
    // segment ends of the tile: bit e set if edge e closes its segment
    const int le = lane < TE ? lane : TE - 1, ln = le + 1 < TE ? le + 1 : le;
    const uint64_t endmask = __ballot(lane < nvalid && (lane == nvalid - 1 || s.seg[ln] != s.seg[le]));
    const int col = cb * CB + 16 * (lane >> 5);  // the lane's first channel
    if constexpr (P::GW) {
      // bias and pre-activation rows; the gate values through the stages (every
      // wave passes both barriers); the activation; the stores
      static_for<L + 1>([&](auto LO) {
        constexpr int lo = decltype(LO)::value;
        if constexpr (P::tab.owner[lo] == W) {
          add_bias<lo>(acc, a, col);
          if (a.gsave != nullptr) save_pre<lo>(acc, s, a, col, lane);
        }
      });
      gate_rows<W>(acc, s, a, col, lane);
      gate_out<W>(acc, st0, st1, st2, lane);
      __syncthreads();
      static_for<L + 1>([&](auto LO) {
        constexpr int lo = decltype(LO)::value;
        if constexpr (P::tab.owner[lo] == W) gate_act_gw<lo>(acc, st0, st1, st2, lane);
      });
      __syncthreads();  // gate values read before the stages are staging again
      static_for<L + 1>([&](auto LO) {
        constexpr int lo = decltype(LO)::value;
        if constexpr (P::tab.owner[lo] == W) {
          if constexpr (MODE == FWD_EDGE)
            save_pre<lo, true>(acc, s, a, col, lane);
          else
            rotate_sum<W, lo>(acc, s, a, cb, buf, lane, endmask);
        }
      });
      return;
    }
    static_for<L + 1>([&](auto LO) {
      constexpr int lo = decltype(LO)::value;
      if constexpr (P::tab.owner[lo] == W) {
        if constexpr (!P::BWD) {
          add_bias<lo>(acc, a, col);
          if constexpr (GATE) {
            if (a.gsave != nullptr) save_pre<lo>(acc, s, a, col, lane);
            gate_act<lo>(acc);
          }
        } else if constexpr (RAD)
          radial<lo>(acc, s, a, col, lane);
        if constexpr (MODE == BWD_EDGE)
          store_gate_bwd<lo>(acc, s, a, col, lane);
        else if constexpr (MODE == FWD_EDGE)
          save_pre<lo, true>(acc, s, a, col, lane);
        else
          rotate_sum<W, lo>(acc, s, a, cb, buf, lane, endmask);
      }
    });
  }

  template <int W, int KR, bool RAD>
  static __device__ __forceinline__ void body(Smem& s, char* st0, char* st1, char* st2,
                                              const Args& a,
                                              int cb, int tid, int nvalid) {
    const int wave = tid >> 6, lane = tid & 63;
    f32x16 acc[P::MSLOT];
#pragma unroll
    for (int k = 0; k < P::MSLOT; ++k)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[k][i] = 0.f;

    const int nks = a.C_k / KC;
    const char* wp = a.wpack + static_cast<int64_t>(cb) * a.frags_per_cb * FRAG;
    AState st;
    a_init<W>(st, s, a, lane);
    frag_t bn[P::NBW];
    // ring prologue, in the issue order kstep expects: DMA of step 0, B of
    // step 0, DMA of step 1
    a_dma<W, 0>(st, st0, a, 0);
    b_load<W, 0>(bn, wp, 0, 0, lane);
    if constexpr (KR == 3) {
      if constexpr (L >= 1) a_dma<W, (L >= 1 ? 1 : 0)>(st, st1, a, 0);
    } else {
      a_dma<W, 0>(st, st1, a, 1);
    }
    int64_t foff = 0;
    static_for<L + 1>([&](auto LIc) {
      constexpr int LI = decltype(LIc)::value;
      kdegree<W, LI, KR>(acc, bn, st, st0, st1, st2, a, wp, foff, nks, lane);
      foff += static_cast<int64_t>(nks) * P::nbfrag(LI);
    });
    __syncthreads();  // all A reads done before the stages become epilogue staging
    epilogue<W, RAD>(acc, s, a, cb, lane, nvalid, wave_staging(wave, st0, st1, st2), st0, st1, st2);
  }

  // The tile's edges (e0 .. e0 + nvalid - 1, may be none) and where the segment
  // that ends at each goes: by the tile's threads 0 .. TE - 1, before a barrier.
  // Segments cut by the tile boundary go to the partials buffer: the tile's
  // first segment (slot 0) if it began in an earlier tile, its last one (slot 1)
  // if it continues into the next tile.
  static __device__ __forceinline__ void setup(Smem& s, const Args& a, int64_t tile, int64_t e0, int nvalid, int tid,
                                               int safe) {
    if (tid < TE) {
      int sg = -1, ei = -1;
      float* dst = nullptr;
      if (tid < nvalid) {
        const int64_t p = e0 + tid, el = e0 + nvalid - 1;
        const int s0 = a.seg[e0], s1 = a.seg[el];
        const bool fp = e0 > 0 && a.seg[e0 - 1] == s0;
        const bool lp = el + 1 < a.E && a.seg[el + 1] == s1;
        sg = a.seg[p];
        ei = a.eidx ? a.eidx[p] : static_cast<int>(p);
        const int64_t ow = a.ow > 0 ? a.ow : a.C_n;
        if ((sg == s0 && fp) || (sg == s1 && lp))
          dst = a.part + (tile * 2 + (sg == s0 ? 0 : 1)) * d * ow;
        else
          dst = a.out + static_cast<int64_t>(sg) * d * ow;
      }
      s.seg[tid] = sg;
      s.eid[tid] = ei;
      s.optr[tid] = dst;
    }
    if (tid == 0) s.safe = safe;
  }

  template <int KR, bool RAD>
  static __device__ __forceinline__ void run(const Args& a) {
    __shared__ Smem s;
    __shared__ alignas(16) char st0[SB];
    __shared__ alignas(16) char st1[SB];
    __shared__ alignas(16) char st2[SB];
    const int tid = threadIdx.x, wave = tid >> 6;
    // XCD-aware mapping: consecutive workgroup ids go round-robin over the 8
    // XCDs.  The n_cb channel-block workgroups of one edge tile are the
    // consecutive workgroups of one XCD, so they run together and read the
    // tile's rows from that XCD's L2 (each XCD holds the weights of all blocks).
    const int64_t bid = blockIdx.x;
    const int64_t slot = bid >> 3;
    const int cb = a.cb0 + static_cast<int>(slot % a.n_cb);
    const int64_t tile = (slot / a.n_cb) * 8 + (bid & 7);
    if (tile >= a.ntiles) return;  // whole workgroup exits together
    const int64_t e0 = tile * TE;
    const int nvalid = static_cast<int>((a.E - e0) < TE ? (a.E - e0) : TE);
    setup(s, a, tile, e0, nvalid, tid, a.eidx ? a.eidx[e0] : static_cast<int>(e0));
    __syncthreads();
    static_for<NW>([&](auto WI) {
      constexpr int w = decltype(WI)::value;
      if (wave == w) body<w, KR, RAD>(s, st0, st1, st2, a, cb, tid, nvalid);
    });
  }
};

// KR: (C_k / KC) % 3 if C_k / KC >= 2, else 3.
// RAD (input gradient only): a radial scale is given (its gradient is formed).
// MINB: resident workgroups per CU the register allocation targets.
template <int L, int M, bool GATE, int NW, int RT, class TM, int MODE, int KR, bool RAD, int MINB>
__global__ __launch_bounds__(NW * 64, MINB) void gemm_kernel(Args a) {
  Gemm<L, M, GATE, NW, RT, TM, MODE>::template run<KR, RAD>(a);
}

}  // namespace msg
}  // namespace maloq
