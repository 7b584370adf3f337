// gqa_flat.hpp — how a flat split (SplitParams::slots) cuts a batch: the walk
// of one slot over its pieces, and the combine's plan.  Written against a wave
// type W (gqa_decode.hip's on the GPU; an array of 64 lanes in the host test),
// since the lengths of a paged batch live on the device and every wave works
// its range out for itself.
//
// W: B, slots, seq_units (contiguous: units per sequence); Lanes, one int per
// lane; units(base, keys): per lane, the units and keys of sequence base +
// lane; scan: inclusive sum over the lanes; add: lane by lane; read(v, l):
// lane l's value; first_above(v, x): first lane whose value exceeds x; share(n)
// = n / slots, sequence(n) = n / seq_units; own(v, lane): the value of `lane`;
// each(f): f(lane) for every lane of the caller.
#pragma once

#if defined(__HIPCC__)
#define GQA_WAVE_FN __device__ __forceinline__
#else
#define GQA_WAVE_FN inline
#endif

namespace gqa {

// The pieces of one slot: ranges of consecutive tile steps ("units") of one
// sequence each, in order.  The slot's range is [j * T / slots, (j + 1) * T /
// slots) of the T units of all sequences (with fewer units than slots, unit j
// alone, so that no slot between two pieces of a sequence is empty).  Every
// value is wave-uniform except the Lanes.
template <class W, bool PAGED> struct FlatWalk {
  using Lanes = typename W::Lanes;
  int at, end;      // units of the flat order still to do
  int b, u0, n;     // current sequence, its first unit in the flat order, its units
  int base, carry;  // paged: first sequence of the scanned group of 64, units before it
  Lanes incl, mine, keys;  // paged: scan over the group; its sequences' units and keys
  int skv;          // paged: keys of the current sequence

  GQA_WAVE_FN void scan(const W& w) {
    mine = w.units(base, keys);
    incl = W::scan(mine);
  }
  GQA_WAVE_FN static int total_of(const W& w, int from) {
    Lanes sum{}, k;
    for (int g0 = from; g0 < w.B; g0 += 64) W::add(sum, w.units(g0, k));
    return W::read(W::scan(sum), 63);
  }

  GQA_WAVE_FN void start(const W& w, int slot) {
    int total;
    if constexpr (PAGED) {
      base = 0;
      carry = 0;
      scan(w);
      total = W::read(incl, 63);
      if (w.B > 64) total += total_of(w, 64);
    } else {
      n = w.seq_units;
      total = n * w.B;
    }
    if (total < w.slots) {
      at = slot < total ? slot : total;
      end = slot + 1 < total ? slot + 1 : total;
    } else {
      at = w.share(slot * total);
      end = w.share((slot + 1) * total);
    }
    if constexpr (PAGED) {
      b = 0;
      u0 = 0;
      n = 0;
    } else if (at < end) {
      b = w.sequence(at);
      u0 = b * n;
    }
  }

  // The next piece: units [from, from + cnt) of sequence b.  With more than 64
  // sequences the lengths are read again as the walk reaches them; a caller
  // that shortens them meanwhile gets a walk that ends with the batch.
  GQA_WAVE_FN bool next(const W& w, int& from, int& cnt) {
    if (at >= end) return false;
    if constexpr (PAGED) {
      while (at >= carry + W::read(incl, 63)) {
        if (base + 64 >= w.B) return false;
        carry += W::read(incl, 63);
        base += 64;
        scan(w);
      }
      const int l = W::first_above(incl, at - carry);
      b = base + l;
      n = W::read(mine, l);
      skv = W::read(keys, l);
      u0 = carry + W::read(incl, l) - n;
    } else if (at >= u0 + n) {
      ++b;
      u0 += n;
    }
    from = at - u0;
    cnt = (end < u0 + n ? end : u0 + n) - at;
    at += cnt;
    return true;
  }

  // Paged: put(sequence, first partial, number of partials) for the combine,
  // by one wave: unit t lies in slot ((t + 1) * slots - 1) / T.  Lengths that
  // change between its two reads may not lead past the last partial.
  // (Contiguous sequences are equally long: the combine works it out.)
  template <class Put> GQA_WAVE_FN static void plan(const W& w, Put put) {
    const int total = total_of(w, 0);
    const int slots = w.slots < total ? w.slots : total;
    int before = 0;
    Lanes k;
    for (int g0 = 0; g0 < w.B; g0 += 64) {
      const Lanes m = w.units(g0, k), upto = W::scan(m);
      w.each([&](int lane) {
        const int s = g0 + lane, mine = W::own(m, lane), u1 = before + W::own(upto, lane);
        if (s >= w.B) return;
        int first = 0, count = 0;
        if (mine > 0 && total > 0) {
          const int lo = ((u1 - mine + 1) * slots - 1) / total, hi = (u1 * slots - 1) / total;
          first = lo < slots - 1 ? lo : slots - 1;
          count = (hi < slots - 1 ? hi : slots - 1) - first + 1;
        }
        put(s, first + s, count);
      });
      before += W::read(upto, 63);
    }
  }
};

}  // namespace gqa
