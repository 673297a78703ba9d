// Load-time choice of the runs of plan steps that become one launch with the activations in LDS
// (cvmhip_resident_launch), and the tables of those launches.
//
// A candidate is any stretch of consecutive steps of kinds the launch knows whose tensors, as far as they are alive
// together, fit in LDS.  For every step an estimate of its time inside such a launch is compared with its time as a launch
// of its own; the stretch that saves most is taken, then the next one among the steps that are left.  The estimates:
//   * as a launch: 3.8 us however small (what such launches measure in a captured graph), or the operations at 900 TOP/s,
//     the most that the per-layer kernels reach on maps of this size;
//   * in LDS: per layer 1800 clocks from barrier to barrier without any work (the layer's head, the first filters, the first
//     operands, the last result), and the largest of the filter's way through one compute unit (30 bytes a clock from the
//     L2, and 64 from LDS), the instructions (4 clocks each, 4 per pixel tile and K step, 40 per tile for the result, over
//     four SIMDs) and the latency of the K steps behind one another; rounds of
//     workgroups when there are more images than compute units.
// Measured on ResNet-20: 38 us estimated, 39 us measured.  The tail of SSD-512 (10 x 10 maps and smaller, filters of
// 300 KB and more) was 32 us in one launch and the same as single ones: one compute unit reads a filter too slowly.
// ResNet-50's 7 x 7 layers at batch 50 lost 300 us with the single launches estimated at 350 TOP/s.
#include <algorithm>
#include <climits>
#include <cstring>
#include <map>

#include "graph_runtime.h"

namespace cvmrt {

namespace {

const uint32_t kNone = UINT32_MAX;
const int kComputeUnits = 256;

void Check(int rc, const char* what) {
  if (rc == CVMHIP_OK) return;
  if (rc < CVMHIP_ERR_RUNTIME) CVM_VERIFY(false) << what << ": " << cvmhip_last_error();
  CVM_CHECK(false) << what << ": " << cvmhip_last_error();
}

struct DeviceBuffer {
  void* ptr = nullptr;
  ~DeviceBuffer() { if (ptr) cvmhip_free(ptr); }
};

size_t AlignUp(size_t v, size_t a) { return (v + a - 1) / a * a; }
int Pad(int c) { return c <= 16 ? 16 : (c + 31) / 32 * 32; }
int ConvOut(int h, int k, int s, int p, int d) { return (h + 2 * p - (d * (k - 1) + 1)) / s + 1; }

// clocks of one convolution for one image inside the launch
double ConvClocks(int c, int oc, int oh, int ow, int kh, int kw) {
  const double ksteps = (kh * kw * Pad(c) + 191) / 192 * 3, oct = Pad(oc) / 16, ptiles = (oh * ow + 15) / 16;
  const double tiles = oct * ptiles, per_item = tiles >= 64 ? 4 : tiles >= 32 ? 2 : 1;
  const double groups = std::max(1.0, ptiles / per_item);
  const double stream = oct * ksteps * (1024.0 / 30 + (groups - 1) * 1024 / 64);
  const double issue = std::max(1.0, tiles / 4) * (ksteps * 4 + 40) * 4;
  return 1800 + std::max({stream, issue, ksteps * 100});
}

struct Tensor {
  cvmhip_resident_map map{};
  int first = 0, last = 0;   // layers between which it is alive
  size_t bytes() const { return cvmhip_resident_tensor_bytes(map.c, map.h, map.w, map.border_y, map.border_x); }
};

}  // namespace

// What a stretch [first, last] of the plan needs: the layers in order, with tensors by number instead of LDS offsets.
struct HipGraphRuntime::ResidentDraft {
  struct Layer {
    cvmhip_resident_desc d{};
    int src = -1, res = -1, dst = -1;   // tensor numbers
    size_t step = 0;
  };
  std::vector<Layer> layers;
  std::vector<Tensor> tensors;
  size_t lds = 64;
  bool ok = false;
};

double HipGraphRuntime::ResidentGain(const PlanStep& st) const {
  const double rounds = (st.n + kComputeUnits - 1) / kComputeUnits;
  const double us = 1.0 / 2300;   // shader clock inside such kernels
  switch (st.kind) {
    case PlanStep::STEMPACK:
      return 2.7 - rounds * us * (1500 + 40.0 * st.c * ((st.h * st.w + 1023) / 1024));
    case PlanStep::SUM:
      return 3.0 - rounds * us * (900 + 16.0 * (Pad(st.c) / 64 + 1) * (20 * ((st.h + 63) / 64) + 60));
    case PlanStep::POOL: {
      const double items = (st.oh * st.ow * (Pad(st.c) / 4) + 1023) / 1024;
      return 3.5 - rounds * us * (900 + items * 16 * 14 * st.kh * st.kw);
    }
    default: {
      const int oh = ConvOut(st.h, st.kh, st.sh, st.ph, st.dh), ow = ConvOut(st.w, st.kw, st.sw, st.pw, st.dw);
      double alone = std::max(3.8, 2.0 * st.n * oh * ow * st.oc * st.c * st.kh * st.kw / 9e8);
      double clocks = ConvClocks(st.c, st.oc, oh, ow, st.kh, st.kw);
      if (st.pool3) clocks += 900 + ((st.oh * st.ow * (Pad(st.oc) / 4) + 1023) / 1024) * 16 * 14 * 9;
      if (st.pool2) clocks += 900 + (((oh / 2) * (ow / 2) * (Pad(st.oc) / 4) + 1023) / 1024) * 16 * 14 * 4;
      if (st.pool3) alone = std::max(alone, 5.0);
      return alone - rounds * us * clocks;
    }
  }
}

bool HipGraphRuntime::ResidentEligible(const PlanStep& st) const {
  auto fits = [](int c, int h, int w) {
    const size_t b = cvmhip_resident_tensor_bytes(c, h, w, 0, 0);
    return b > 0 && b < cvmhip_resident_lds_limit();
  };
  if (st.n < 1) return false;
  switch (st.kind) {
    case PlanStep::STEMPACK:
      return PacksStagedInput(st) && fits(st.c, st.h, st.w);
    case PlanStep::SUM:
      return fits(st.c, 1, 1);
    case PlanStep::POOL:
      return fits(st.c, st.h, st.w) && fits(st.c, st.oh, st.ow);
    case PlanStep::CONV: {
      if (st.nhwc || st.flat || st.wsrc == kNone) return false;
      const int oh = ConvOut(st.h, st.kh, st.sh, st.ph, st.dh), ow = ConvOut(st.w, st.kw, st.sw, st.pw, st.dw);
      return fits(st.c, st.h, st.w) && oh >= 1 && ow >= 1 && fits(st.oc, oh, ow) && (st.kh - 1) * st.dh < 255 && (st.kw - 1) * st.dw < 255;
    }
    default:
      return false;
  }
}

HipGraphRuntime::ResidentDraft HipGraphRuntime::DraftResident(size_t first, size_t last) const {
  ResidentDraft r;
  std::map<const void*, int> where;   // int8 tensor (or packed image) -> tensor number
  auto use = [&](const void* key, int layer) {
    auto it = where.find(key);
    if (it == where.end()) return -1;
    r.tensors[it->second].last = layer;
    return it->second;
  };
  auto make = [&](const void* key, int c, int h, int w, int layer) {
    Tensor t;
    t.map.c = c; t.map.h = h; t.map.w = w;
    t.first = t.last = layer;
    r.tensors.push_back(t);
    const int number = static_cast<int>(r.tensors.size()) - 1;
    if (key) where[key] = number;
    return number;
  };
  // the map a layer writes
  auto shape = [](cvmhip_resident_desc* d, int c, int h, int w) {
    d->dst.at = d->src.at = d->res.at = -1;
    d->dst.c = c; d->dst.h = h; d->dst.w = w;
    d->kh = d->kw = d->sh = d->sw = d->dh = d->dw = 1;
  };
  auto window = [](cvmhip_resident_desc* d, int kh, int kw, int sh, int sw, int ph, int pw) {
    d->kh = kh; d->kw = kw; d->sh = sh; d->sw = sw; d->ph = ph; d->pw = pw;
  };
  // an int8 tensor from memory, loaded where it is first needed
  auto load = [&](const void* key, int c, int h, int w, size_t step) {
    const int layer = static_cast<int>(r.layers.size());
    ResidentDraft::Layer l;
    l.d.kind = 1;
    shape(&l.d, c, h, w);
    l.d.in = key;
    l.step = step;
    l.dst = make(key, c, h, w, layer);
    r.layers.push_back(l);
  };
  // does a step outside the stretch, or a later one inside it, read this tensor?
  auto readers = [&](const void* key, size_t producer, bool* inside, bool* outside) {
    *inside = *outside = false;
    for (size_t k = 0; k < plan_.size(); ++k) {
      const PlanStep& st = plan_[k];
      if (st.kind == PlanStep::NODE || st.kind == PlanStep::PACK || st.kind == PlanStep::STEMPACK || st.stem) continue;
      if (!ReadsI8(st, key)) continue;
      if (k < first || k > last) *outside = true;
      else if (k > producer) *inside = true;
    }
  };
  auto finish = [&](ResidentDraft::Layer l, const PlanStep& st, size_t step, bool i8, const void* key, void* out32) {
    const int layer = static_cast<int>(r.layers.size());
    if (i8) {
      bool inside = false, outside = false;
      readers(key, step, &inside, &outside);
      if (outside || !inside) {
        l.d.out_mode = 1;
        l.d.out = const_cast<void*>(key);
      }
      if (inside) l.dst = make(key, l.d.dst.c, l.d.dst.h, l.d.dst.w, layer);
    } else {
      l.d.out_mode = 2;
      l.d.out = out32;
    }
    r.layers.push_back(l);
  };
  for (size_t k = first; k <= last; ++k) {
    const PlanStep& st = plan_[k];
    ResidentDraft::Layer l;
    l.step = k;
    if (st.kind == PlanStep::STEMPACK) {
      // the packed image exists in LDS only: its reader is part of the stretch (a second convolution over the input has a
      // packing step of its own, which the stretch may end with)
      bool inside = false, outside = false;
      for (size_t q = 0; q < plan_.size(); ++q)
        if (plan_[q].stem && plan_[q].aux == st.aux) (q > k && q <= last ? inside : outside) = true;
      if (!inside || outside) return r;
      l.d.kind = 0;
      shape(&l.d, st.c, st.h, st.w);
      l.d.in = in_stage_dev_;
      l.d.range = data_range_;
      l.dst = make(st.aux.get(), st.c, st.h, st.w, static_cast<int>(r.layers.size()));
      r.layers.push_back(l);
      continue;
    }
    const void* src = st.stem ? static_cast<const void*>(st.aux.get()) : i8_ptr_[st.src];
    if (!where.count(src)) {
      if (st.stem) return r;   // its packed image belongs to a step in front of the stretch
      // (a sum's own extent is its pixels in a row, but other layers may read the map as well)
      const bool sum = st.kind == PlanStep::SUM;
      load(src, st.c, sum ? static_cast<int>(shape_[st.src][2]) : st.h, sum ? static_cast<int>(shape_[st.src][3]) : st.w, k);
    }
    const void* res = st.kind == PlanStep::CONV && st.src2 != kNone ? i8_ptr_[st.src2] : nullptr;
    const int oh = st.kind == PlanStep::CONV ? ConvOut(st.h, st.kh, st.sh, st.ph, st.dh) : st.oh;
    const int ow = st.kind == PlanStep::CONV ? ConvOut(st.w, st.kw, st.sw, st.pw, st.dw) : st.ow;
    if (res && !where.count(res)) load(res, st.oc, oh, ow, k);
    const int layer = static_cast<int>(r.layers.size());
    l.src = use(src, layer);
    if (res) l.res = use(res, layer);
    void* out32 = st.out_i8 ? nullptr : entry_ptr_[st.dst];
    const void* key = st.kind == PlanStep::POOL || st.out_i8 ? i8_ptr_[st.dst] : nullptr;
    if (st.kind == PlanStep::SUM) {
      l.d.kind = 3;
      shape(&l.d, st.c, 1, 1);
      l.d.chain = st.chain;
      finish(l, st, k, st.out_i8, key, out32);
    } else if (st.kind == PlanStep::POOL) {
      l.d.kind = 4;
      shape(&l.d, st.c, st.oh, st.ow);
      window(&l.d, st.kh, st.kw, st.sh, st.sw, st.ph, st.pw);
      finish(l, st, k, true, key, nullptr);
    } else {
      l.d.kind = 2;
      shape(&l.d, st.oc, oh, ow);
      window(&l.d, st.kh, st.kw, st.sh, st.sw, st.ph, st.pw);
      l.d.dh = st.dh;
      l.d.dw = st.dw;
      r.tensors[l.src].map.border_y = std::max(r.tensors[l.src].map.border_y, st.ph);
      r.tensors[l.src].map.border_x = std::max(r.tensors[l.src].map.border_x, st.pw);
      l.d.chain = st.chain;
      if (res) l.d.chain2 = st.chain2;
      if (st.pool2 || st.pool3) {
        l.dst = make(nullptr, st.oc, oh, ow, layer);
        r.tensors[l.dst].last = layer + 1;
        const int between = l.dst;
        r.layers.push_back(l);
        ResidentDraft::Layer p;
        p.step = k;
        p.src = between;
        p.d.kind = 4;
        if (st.pool3) {
          shape(&p.d, st.oc, st.oh, st.ow);
          window(&p.d, 3, 3, 2, 2, 1, 1);
        } else {
          shape(&p.d, st.oc, oh / 2, ow / 2);
          window(&p.d, 2, 2, 2, 2, 0, 0);
        }
        finish(p, st, k, true, key, nullptr);
      } else {
        finish(l, st, k, st.out_i8, key, out32);
      }
    }
  }
  // maps of one extent get one border, so that a map over an earlier one's place finds it zero
  for (Tensor& x : r.tensors)
    for (const Tensor& y : r.tensors)
      if (x.map.c == y.map.c && x.map.h == y.map.h && x.map.w == y.map.w) {
        x.map.border_y = std::max(x.map.border_y, y.map.border_y);
        x.map.border_x = std::max(x.map.border_x, y.map.border_x);
      }
  // first fit in order of birth; a layer's operands and its result are alive together
  for (size_t t = 0; t < r.tensors.size(); ++t) {
    Tensor& x = r.tensors[t];
    const size_t size = x.bytes();
    if (size == 0) return r;
    size_t at = 0;
    for (bool moved = true; moved;) {
      moved = false;
      for (size_t u = 0; u < t; ++u) {
        const Tensor& y = r.tensors[u];
        const bool together = x.first <= y.last && y.first <= x.last;
        const size_t from = static_cast<size_t>(y.map.at), to = from + y.bytes();
        if (together && at < to && from < at + size) {
          at = (to + 15) & ~static_cast<size_t>(15);
          moved = true;
        }
      }
    }
    x.map.at = static_cast<int>(at);
    r.lds = std::max(r.lds, at + size);
  }
  // a map over the exact place of an earlier one, with nothing else there in between, finds that one's border
  for (ResidentDraft::Layer& l : r.layers) {
    if (l.dst < 0) continue;
    const Tensor& x = r.tensors[l.dst];
    const Tensor* before = nullptr;
    for (const Tensor& y : r.tensors) {
      const size_t from = static_cast<size_t>(y.map.at), at = static_cast<size_t>(x.map.at);
      if (&y != &x && y.first < x.first && at < from + y.bytes() && from < at + x.bytes() && (!before || y.first > before->first)) before = &y;
    }
    l.d.border_clean = before && std::memcmp(&before->map, &x.map, sizeof(x.map)) == 0 ? 1 : 0;
  }
  // behind the maps two places for filters, which the convolutions take in turn
  size_t need[2] = {0, 0};
  int convs = 0;
  for (const ResidentDraft::Layer& l : r.layers) {
    if (l.d.kind != 2) continue;
    const PlanStep& st = plan_[l.step];
    size_t& most = need[convs++ & 1];
    most = std::max(most, cvmhip_resident_filter_bytes(st.oc, st.c, st.kh, st.kw, l.d.dst.h, l.d.dst.w));
  }
  const size_t filters = (r.lds + 15) & ~static_cast<size_t>(15);
  convs = 0;
  for (ResidentDraft::Layer& l : r.layers)
    if (l.d.kind == 2) l.d.filter_at = static_cast<int>(filters + (convs++ & 1 ? need[0] : 0));
  r.lds = filters + need[0] + need[1];
  r.ok = r.lds <= cvmhip_resident_lds_limit();
  return r;
}

void HipGraphRuntime::BuildResident() {
  resident_at_.assign(plan_.size(), -1);
  in_resident_.assign(plan_.size(), false);
  if (!hooks_.resident) return;
  const size_t n = plan_.size();
  std::vector<double> gain(n, 0);
  std::vector<bool> ok(n, false);
  for (size_t i = 0; i < n; ++i) {
    ok[i] = ResidentEligible(plan_[i]);
    if (ok[i]) gain[i] = ResidentGain(plan_[i]);
  }
  for (;;) {
    double best = 3.0;   // less is within what the estimates are worth
    size_t from = 0, to = 0;
    for (size_t i = 0; i < n; ++i) {
      double sum = -2.0;   // the launch itself, and its first operands
      for (size_t j = i; j < n && ok[j] && !in_resident_[j] && plan_[j].n == plan_[i].n; ++j) {
        sum += gain[j];
        if (j == i || sum <= best) continue;
        if (!DraftResident(i, j).ok) continue;
        best = sum;
        from = i;
        to = j;
      }
    }
    if (to == from) break;
    ResidentDraft d = DraftResident(from, to);
    ResidentRun r;
    r.first = from;
    r.last = to;
    r.nlayers = static_cast<int>(d.layers.size());
    r.images = plan_[from].n;
    r.lds = d.lds;
    std::vector<char> table(d.layers.size() * cvmhip_resident_layer_bytes());
    // filters and table in one allocation: a layer's first touch of pages of its own is a trip to the page tables
    size_t total = AlignUp(table.size(), 256);
    std::vector<size_t> filter_at(d.layers.size(), 0);
    for (size_t l = 0; l < d.layers.size(); ++l) {
      if (d.layers[l].d.kind != 2) continue;
      const PlanStep& st = plan_[d.layers[l].step];
      filter_at[l] = total;
      total += cvmhip_resident_filter_bytes(st.oc, st.c, st.kh, st.kw, d.layers[l].d.dst.h, d.layers[l].d.dst.w);
    }
    auto buf = std::make_shared<DeviceBuffer>();
    Check(cvmhip_alloc(&buf->ptr, total), "resident run");
    char* base = static_cast<char*>(buf->ptr);
    std::vector<char> places(total);
    for (size_t l = 0; l < d.layers.size(); ++l) {
      ResidentDraft::Layer& layer = d.layers[l];
      const PlanStep& st = plan_[layer.step];
      if (layer.src >= 0) layer.d.src = d.tensors[layer.src].map;
      if (layer.res >= 0) layer.d.res = d.tensors[layer.res].map;
      if (layer.dst >= 0) layer.d.dst = d.tensors[layer.dst].map;
      if (layer.d.kind == 2) {
        void* filter = base + filter_at[l];
        Check(cvmhip_resident_pack_filter(entry_ptr_[st.wsrc], st.bias, filter, st.oc, st.c, st.kh, st.kw, st.dh, st.dw,
                                          layer.d.src.w + 2 * layer.d.src.border_x, stream_), "resident filter");
        layer.d.filter = filter;
        const double work = static_cast<double>(st.oc) * st.c * st.kh * st.kw;
        r.ops += 2.0 * r.images * layer.d.dst.h * layer.d.dst.w * work;
        r.bytes += work;
      }
      size_t bytes = 0, off = 0;
      Check(cvmhip_resident_layer(table.data(), static_cast<int>(l), &layer.d, places.data(), &bytes, &off), "resident layer");
      if (bytes > 0) {
        Check(cvmhip_copy_h2d(base + filter_at[l] + off, places.data(), bytes, stream_), "resident places");
        Check(cvmhip_stream_sync(stream_), "resident places");   // the buffer is used again
      }
    }
    Check(cvmhip_copy_h2d(base, table.data(), table.size(), stream_), "resident table");
    Check(cvmhip_stream_sync(stream_), "resident table");   // the host copy goes away
    const ResidentDraft::Layer& tail = d.layers.back();
    r.whole_call = from == 0 && to + 1 == n && outputs_.size() == 1 && tail.d.out_mode == 2 && tail.d.out == entry_ptr_[entry_id(outputs_[0])];
    for (size_t l = 0; l < d.layers.size(); ++l)
      r.whole_call = r.whole_call && d.layers[l].d.kind != 1 && (l == 0) == (d.layers[l].d.kind == 0) && (d.layers[l].d.out_mode == 0 || l + 1 == d.layers.size());
    r.table = base;
    r.owner = buf;
    resident_at_[from] = static_cast<int>(residents_.size());
    for (size_t k = from; k <= to; ++k) in_resident_[k] = true;
    residents_.push_back(r);
  }
}

}  // namespace cvmrt
