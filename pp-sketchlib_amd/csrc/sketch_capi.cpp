// Sketching entry points (include/ppsk.h, ppsk_sketch / ppsk_sketch_ex):
// work units, device buffers and the launches of sketch_kernels.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "capi_common.h"
#include "sketch_kernels.h"

using namespace ppsk::capi;

namespace {

constexpr int64_t UNIT = 1024;          // most k-mer start positions per lane
constexpr int64_t GROUP_UNITS = 1024;   // most units per workgroup task

// Consecutive parts of the call's buffer, each at a multiple of 256 bytes.
struct Parts {
  size_t used = 0;
  size_t take(size_t bytes) {
    const size_t at = used;
    used += (std::max<size_t>(bytes, 1) + 255) / 256 * 256;
    return at;
  }
};

// Window starts per lane of a hashing launch over `slots` workgroups resident
// at once, for `windows` windows of `pieces` (contig, k) pairs in `jobs`
// (sample, k) pairs.  Units of UNIT windows give the least rolling-in (k - 1
// steps per unit), but a launch that fits the slots in one round must spread
// over all of them: the smallest unit of at least 64 windows whose groups (one
// unit per lane; at most windows / unit + pieces units, the last group of a job
// partly filled) need no second round.  6 genomes of 2 Mb at 8 k-mer lengths: 96
// groups of 1,024-window units on 512 slots took 494 us, 480 groups of 416 take
// 207.
int64_t unit_windows(int64_t windows, int64_t pieces, int64_t jobs, int64_t slots) {
  const int64_t lanes = (slots - jobs) * ppsk::SKETCH_TB - pieces;
  if (lanes <= 0 || windows > lanes * UNIT) return UNIT;
  return std::min(UNIT, std::max<int64_t>(64, ((windows + lanes - 1) / lanes + 15) / 16 * 16));
}

// contigs: the contigs of contig_off wherever they lie, or null: one after the
// other in seq.
int sketch_impl(int device_id, int64_t n_samples, const char* seq, int64_t seq_bytes,
                const char* const* contigs, const int64_t* contig_off, int64_t n_contigs, const int64_t* sample_contig,
                int32_t n_k, const int32_t* klist, int32_t sketchsize64, int32_t use_rc,
                int32_t codon, int32_t min_count, int32_t exact, uint64_t* raw_out,
                double* inv_minhash, int32_t* densified) {
  if (n_samples < 1 || !sample_contig || !raw_out) {
    return fail(PPSK_ERR_ARG, "sketching needs at least one sample and an output buffer");
  }
  if (n_contigs < 0 || (n_contigs > 0 && (!contig_off || (!seq && !contigs)))) {
    return fail(PPSK_ERR_ARG, "contig offsets / sequence missing");
  }
  if (n_k < 1 || n_k > ppsk::MAXK || !klist) {
    return fail(PPSK_ERR_ARG, "n_k must be in [1, " + std::to_string(ppsk::MAXK) + "]");
  }
  for (int i = 0; i < n_k; ++i) {
    if (klist[i] < 3) return fail(PPSK_ERR_ARG, "Minimum k must be 3 or higher");
    if ((codon ? 3 * klist[i] : klist[i]) > ppsk::SKETCH_MAX_K) {
      return fail(PPSK_ERR_ARG, "k must be at most " +
                                    std::to_string(ppsk::SKETCH_MAX_K / (codon ? 3 : 1)));
    }
    if (i && klist[i] <= klist[i - 1]) return fail(PPSK_ERR_ARG, "klist must be strictly ascending");
  }
  if (sketchsize64 < 1 || sketchsize64 > 1023) {
    return fail(PPSK_ERR_ARG, "sketchsize64 must be in [1, 1023]");
  }
  if (min_count < 0 || min_count > 255) return fail(PPSK_ERR_ARG, "min_count must be in [0, 255]");
  if (sample_contig[0] != 0 || sample_contig[n_samples] != n_contigs) {
    return fail(PPSK_ERR_ARG, "sample_contig must run from 0 to n_contigs");
  }
  for (int64_t s = 0; s < n_samples; ++s) {
    if (sample_contig[s + 1] < sample_contig[s]) return fail(PPSK_ERR_ARG, "sample_contig not ascending");
  }
  for (int64_t c = 0; c < n_contigs; ++c) {
    if (contig_off[c + 1] < contig_off[c] || contig_off[c + 1] > seq_bytes || contig_off[c] < 0) {
      return fail(PPSK_ERR_ARG, "contig offsets outside the sequence buffer");
    }
  }
  // windows span k bases, or 3k - 2 with codon-phased seeds
  auto span = [codon](int32_t k) -> int64_t { return codon ? 3 * (int64_t)k - 2 : k; };
  const bool filtered = min_count > 0;
  if (filtered) {
    for (int64_t s = 0; s < n_samples; ++s) {
      int64_t w = 0;
      for (int64_t ci = sample_contig[s]; ci < sample_contig[s + 1]; ++ci) {
        w += std::max<int64_t>(0, contig_off[ci + 1] - contig_off[ci] - span(klist[0]) + 1);
      }
      if (w > ppsk::READS_MAX_WINDOWS) {
        return fail(PPSK_ERR_ARG, "a sample has more than " +
                                      std::to_string(ppsk::READS_MAX_WINDOWS) +
                                      " k-mer windows for count filtering");
      }
    }
  }
  DeviceCtx* c = nullptr;
  if (int rc = get_ctx(device_id, &c)) return rc;
  std::lock_guard<std::mutex> lk(c->mu);

  const int64_t nbins = (int64_t)sketchsize64 * 64;
  const uint64_t sign_mod = (1ULL << 61) - 1ULL;
  ppsk::SketchArgs a;
  std::memset(&a, 0, sizeof(a));
  a.n_k = n_k;
  a.s64 = sketchsize64;
  a.use_rc = use_rc ? 1 : 0;
  a.codon = codon ? 1 : 0;
  a.n_samples = n_samples;
  a.binsize = (sign_mod + (uint64_t)nbins - 1ULL) / (uint64_t)nbins;
  a.bin_recip = ~0ULL / a.binsize;
  if (a.bin_recip >> 32) return fail(PPSK_ERR_ARG, "bin reciprocal out of range");
  {
    // 2^t = q binsize + r, t from 0 until q has 32 bits (q < 2^16 at t = 61)
    uint64_t q = 0, r = 1;
    int t = 0;
    while ((q >> 31) == 0) {
      q <<= 1;
      r <<= 1;
      if (r >= a.binsize) {
        r -= a.binsize;
        ++q;
      }
      ++t;
    }
    a.bin_g = (uint32_t)q;
    a.bin_s = t - 61;
  }

  // Work units: every contig of every k cut into runs of windows; before_u and
  // before_w count the units and windows of the (k, contig) pairs before each,
  // k by k (index kk * n_contigs + contig).  The unit lists are written from
  // them on the device (launch_sketch_units).
  int64_t unit = UNIT;
  bool lds_bins = false;
  std::vector<int64_t> spans;
  for (int kk = 0; kk < n_k; ++kk) spans.push_back(span(klist[kk]));
  if (!filtered) {
    // bin minima in LDS when one sample's bins fit a workgroup's LDS (the step
    // table takes another 400 bytes)
    int lds = 0;
    HIP_TRY(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device_id));
    lds_bins = (size_t)nbins * sizeof(uint64_t) + 512 <= (size_t)lds;
    int slots = 0;
    HIP_TRY(ppsk::sketch_hash_slots(a, lds_bins, &slots));
    const int64_t bases = n_contigs > 0 ? contig_off[n_contigs] - contig_off[0] : 0;
    unit = unit_windows(bases * n_k, n_contigs * n_k, n_samples * n_k, slots);
  }
  const size_t pieces = (size_t)n_contigs * n_k;
  std::vector<int64_t> before_u(pieces + 1), before_w(pieces + 1);
  {
    int64_t nu = 0, nw = 0;
    size_t f = 0;
    for (int kk = 0; kk < n_k; ++kk) {
      for (int64_t c0 = 0; c0 < n_contigs; ++c0, ++f) {
        before_u[f] = nu;
        before_w[f] = nw;
        const int64_t w = contig_off[c0 + 1] - contig_off[c0] - spans[kk] + 1;
        if (w <= 0) continue;
        nw += w;
        nu += w <= unit ? 1 : (w + unit - 1) / unit;
      }
    }
    before_u[f] = nu;
    before_w[f] = nw;
  }
  // unfiltered: groups (runs of units of one sample and one k) of one hashing
  // launch; filtered: the units and windows of the largest (sample, k)
  std::vector<ppsk::SketchGroup> groups;
  int64_t list_units = 0, max_w = 0;
  const int64_t per_group = unit < UNIT ? ppsk::SKETCH_TB : GROUP_UNITS;
  for (int kk = 0; kk < n_k; ++kk) {
    for (int64_t s = 0; s < n_samples; ++s) {
      const size_t lo = (size_t)kk * n_contigs + sample_contig[s];
      const size_t hi = (size_t)kk * n_contigs + sample_contig[s + 1];
      const int64_t u0 = before_u[lo], u1 = before_u[hi];
      if (filtered) {
        list_units = std::max(list_units, u1 - u0);
        max_w = std::max(max_w, before_w[hi] - before_w[lo]);
        continue;
      }
      for (int64_t g = u0; g < u1; g += per_group) {
        groups.push_back({g, std::min(u1, g + per_group), (int32_t)s, kk});
      }
    }
  }
  const int64_t total_units = before_u[pieces];
  if (!filtered) list_units = total_units;
  const size_t ws_bytes = filtered ? ppsk::reads_workspace_bytes(max_w) : 0;

  // one buffer for the call, kept with the context up to 1 GiB
  const size_t raw_words = (size_t)n_samples * n_k * sketchsize64 * ppsk::BBITS_SK;
  Parts parts;
  const size_t stats = (size_t)n_samples * n_k;
  // base codes, padded both sides for the kernel's stream loads
  const size_t at_seq = parts.take((size_t)(ppsk::CODE_PAD_FRONT + seq_bytes + ppsk::CODE_PAD_BACK));
  const size_t at_units = parts.take((size_t)list_units * sizeof(ppsk::SketchUnit));
  const size_t at_wbase = parts.take(filtered ? (size_t)list_units * sizeof(int64_t) : 0);
  // contig offsets, spans, before_u, before_w
  const size_t index_words = (size_t)n_contigs + 1 + n_k + (pieces + 1) * (filtered ? 2 : 1);
  const size_t at_index = parts.take(index_words * sizeof(int64_t));
  const size_t at_groups = parts.take(groups.size() * sizeof(ppsk::SketchGroup));
  const size_t at_k = parts.take(n_k * sizeof(int32_t));
  const size_t at_signs = parts.take(stats * nbins * sizeof(uint64_t));
  const size_t at_raw = parts.take(raw_words * sizeof(uint64_t));
  const size_t at_stats = parts.take(stats * (sizeof(double) + sizeof(int32_t)));
  const size_t at_next = parts.take(sizeof(int));
  const size_t at_ws = parts.take(ws_bytes);
  if (int rc = grow(c, &c->sketch, &c->sketch_bytes, parts.used, WS_ALL & ~WS_SKETCH)) return rc;
  struct Trim {
    DeviceCtx* c;
    ~Trim() {
      hipStreamSynchronize(c->stream);  // after an error: nothing may still read the inputs
      trim(&c->sketch, &c->sketch_bytes);
    }
  } trimmed{c};
  char* mem = (char*)c->sketch;
  uint8_t* codes = (uint8_t*)(mem + at_seq) + ppsk::CODE_PAD_FRONT;
  if (contigs) {
    HIP_TRY(fill_device(c, codes, (size_t)seq_bytes, c->stream, [&](char* to, size_t at, size_t n) {
      int64_t ci = std::upper_bound(contig_off, contig_off + n_contigs + 1, (int64_t)at) - contig_off - 1;
      for (size_t done = 0; done < n; ++ci) {
        const size_t from = at + done - (size_t)contig_off[ci];
        const size_t m = std::min(n - done, (size_t)(contig_off[ci + 1] - contig_off[ci]) - from);
        std::memcpy(to + done, contigs[ci] + from, m);
        done += m;
      }
    }));
  } else {
    HIP_TRY(copy_to_device(c, codes, seq, (size_t)seq_bytes, c->stream));
  }
  ppsk::UnitIndex ix;
  ix.contig_off = (const int64_t*)(mem + at_index);
  ix.spans = ix.contig_off + n_contigs + 1;
  ix.before_u = ix.spans + n_k;
  ix.before_w = filtered ? ix.before_u + pieces + 1 : nullptr;
  ix.n_contigs = n_contigs;
  ix.unit = unit;
  if (n_contigs > 0) {
    HIP_TRY(copy_to_device(c, (void*)ix.contig_off, contig_off, (n_contigs + 1) * sizeof(int64_t), c->stream));
  }
  HIP_TRY(copy_to_device(c, (void*)ix.spans, spans.data(), n_k * sizeof(int64_t), c->stream));
  HIP_TRY(copy_to_device(c, (void*)ix.before_u, before_u.data(), (pieces + 1) * sizeof(int64_t), c->stream));
  if (filtered) {
    HIP_TRY(copy_to_device(c, (void*)ix.before_w, before_w.data(), (pieces + 1) * sizeof(int64_t), c->stream));
  }
  HIP_TRY(copy_to_device(c, mem + at_groups, groups.data(),
                         groups.size() * sizeof(ppsk::SketchGroup), c->stream));
  HIP_TRY(copy_to_device(c, mem + at_k, klist, n_k * sizeof(int32_t), c->stream));
  a.codes = codes;
  a.units = (const ppsk::SketchUnit*)(mem + at_units);
  a.groups = (const ppsk::SketchGroup*)(mem + at_groups);
  a.klist = (const int32_t*)(mem + at_k);
  a.signs = (uint64_t*)(mem + at_signs);
  a.raw = (uint64_t*)(mem + at_raw);
  a.inv_minhash = (double*)(mem + at_stats);
  a.densified = (int32_t*)(a.inv_minhash + stats);

  hipEvent_t e0 = pool_event(c, 0), e1 = pool_event(c, 1);
  if (!e0 || !e1) return fail(PPSK_ERR_HIP, "event creation failed");
  HIP_TRY(hipEventRecord(e0, c->stream));
  HIP_TRY(ppsk::launch_sketch_decode(codes, seq_bytes, c->stream));
  int64_t items = 0;
  ppsk::SketchUnit* d_units = (ppsk::SketchUnit*)(mem + at_units);
  int64_t* d_wbase = (int64_t*)(mem + at_wbase);
  if (!filtered) {
    items = total_units;
    HIP_TRY(ppsk::launch_sketch_units(ix, 0, (int64_t)pieces, total_units, d_units, nullptr, c->stream));
    HIP_TRY(ppsk::launch_sketch(a, (int64_t)groups.size(), lds_bins, (int*)(mem + at_next), c->stream));
  } else {
    // one (sample, k) at a time through the counting pipeline
    HIP_TRY(ppsk::launch_sketch_reset(a, c->stream));
    for (int64_t s = 0; s < n_samples; ++s) {
      for (int kk = 0; kk < n_k; ++kk) {
        const int64_t lo = kk * n_contigs + sample_contig[s], hi = kk * n_contigs + sample_contig[s + 1];
        const int64_t nu = before_u[hi] - before_u[lo], nw = before_w[hi] - before_w[lo];
        if (nw == 0) continue;
        HIP_TRY(ppsk::launch_sketch_units(ix, lo, hi, nu, d_units, d_wbase, c->stream));
        ppsk::ReadsJob rj;
        rj.codes = codes;
        rj.units = d_units;
        rj.wbase = d_wbase;
        rj.n_units = nu;
        rj.n_windows = nw;
        rj.k = klist[kk];
        rj.use_rc = use_rc ? 1 : 0;
        rj.min_count = min_count;
        rj.exact = exact ? 1 : 0;
        rj.codon = codon ? 1 : 0;
        rj.binsize = a.binsize;
        rj.recip = (uint32_t)a.bin_recip;
        rj.bins = a.signs + (s * n_k + kk) * nbins;
        rj.words = c->words;
        HIP_TRY(ppsk::run_reads_job(rj, mem + at_ws, ws_bytes, c->stream));
        items += nu;
      }
    }
    HIP_TRY(ppsk::launch_sketch_finish(a, c->stream));
  }
  HIP_TRY(hipEventRecord(e1, c->stream));
  HIP_TRY(copy_to_host(c, raw_out, a.raw, raw_words * sizeof(uint64_t), c->stream));
  std::vector<char> st(stats * (sizeof(double) + sizeof(int32_t)));
  HIP_TRY(copy_to_host(c, st.data(), a.inv_minhash, st.size(), c->stream));
  const double* mh = (const double*)st.data();
  const int32_t* dn = (const int32_t*)(mh + stats);
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
  g_last_ms = ms;
  g_last_launches = 1;
  g_last_items = items;
  for (int64_t s = 0; s < n_samples; ++s) {
    double sum = 0.0;
    int32_t d = 0;
    for (int kk = 0; kk < n_k; ++kk) {
      sum += mh[(size_t)s * n_k + kk];
      d |= dn[(size_t)s * n_k + kk] != 0 ? 1 : 0;
    }
    if (inv_minhash) inv_minhash[s] = sum;
    if (densified) densified[s] = d;
  }
  return PPSK_OK;
}

}  // namespace

extern "C" {

int ppsk_sketch(int device_id, int64_t n_samples, const char* seq, int64_t seq_bytes,
                const int64_t* contig_off, int64_t n_contigs, const int64_t* sample_contig,
                int32_t n_k, const int32_t* klist, int32_t sketchsize64, int32_t use_rc,
                uint64_t* raw_out, double* inv_minhash, int32_t* densified) {
  return sketch_impl(device_id, n_samples, seq, seq_bytes, nullptr, contig_off, n_contigs,
                     sample_contig, n_k, klist, sketchsize64, use_rc, 0, 0, 0, raw_out, inv_minhash,
                     densified);
}

int ppsk_sketch_ex(int device_id, int64_t n_samples, const char* seq, int64_t seq_bytes,
                   const int64_t* contig_off, int64_t n_contigs, const int64_t* sample_contig,
                   int32_t n_k, const int32_t* klist, int32_t sketchsize64, int32_t use_rc,
                   int32_t codon_phased, int32_t min_count, int32_t exact, uint64_t* raw_out,
                   double* inv_minhash, int32_t* densified) {
  return sketch_impl(device_id, n_samples, seq, seq_bytes, nullptr, contig_off, n_contigs,
                     sample_contig, n_k, klist, sketchsize64, use_rc, codon_phased, min_count, exact,
                     raw_out, inv_minhash, densified);
}

int ppsk_sketch_contigs(int device_id, int64_t n_samples, const char* const* contigs,
                        const int64_t* contig_off, int64_t n_contigs, const int64_t* sample_contig,
                        int32_t n_k, const int32_t* klist, int32_t sketchsize64, int32_t use_rc,
                        int32_t codon_phased, int32_t min_count, int32_t exact, uint64_t* raw_out,
                        double* inv_minhash, int32_t* densified) {
  if (n_contigs > 0 && (!contigs || !contig_off)) {
    return fail(PPSK_ERR_ARG, "contig offsets / sequence missing");
  }
  if (n_contigs > 0 && contig_off[0] != 0) return fail(PPSK_ERR_ARG, "contig offsets must start at 0");
  return sketch_impl(device_id, n_samples, nullptr, n_contigs > 0 ? contig_off[n_contigs] : 0, contigs,
                     contig_off, n_contigs, sample_contig, n_k, klist, sketchsize64, use_rc,
                     codon_phased, min_count, exact, raw_out, inv_minhash, densified);
}

}  // extern "C"
