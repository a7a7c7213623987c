// Slices: the first steps of a program run several times over, each time on a part of the leading dimension (a batch's
// images, a matrix's rows), so that the link carries the next part up -- and the part before down -- meanwhile.
#include <algorithm>

#include "hip_planner.h"

namespace pmlc::target::hip {

namespace {

int64_t elemBytes(int32_t dtype) { return static_cast<int64_t>(util::byteSize(static_cast<DataType>(dtype))); }

// What a step reads and writes, taken as `units` of its leading dimension: the buffers that a part of it touches the same
// part of, and those that it reads as they are.
struct Uses {
  std::vector<int> rows, shared, results;
};

class Slicer {
 public:
  Slicer(const Plan& plan, int64_t units) : plan_(plan), units_(units) {}

  // The step on `part` of its units, or false where its parts cannot be told apart.
  bool slice(const Step& s, int64_t part, Step* out, Uses* uses) const {
    *out = s;
    *uses = {};
    if (!s.schedule.empty() || !s.outs.empty() || s.a_off != 0 || s.c_off != 0 || s.a2_off != 0) return false;
    for (int64_t off : s.operand_off)
      if (off != 0) return false;
    switch (s.kind) {
      case Step::Gemm: {
        pml_hip_gemm_desc& d = out->gemm;
        const int64_t m = d.m, es = elemBytes(d.in_dtype);
        if (s.out2 >= 0 && !s.chained) return false;
        if (!share(&d.m, part) || !lies(s.a, m * d.lda * es) || !lies(s.c, m * d.ldc * elemBytes(d.c_dtype))) return false;
        if (d.init_kind && d.init_row_stride != 0) return false;
        uses->rows = {s.a};
        uses->shared = {s.b, s.init};
        uses->results = {s.c};
        if (d.k2 > 0) {
          // (rows of the second left-hand side: one a result row, or the pixels of whole images)
          const int64_t images = d.a2_stride > 0 ? m / std::max<int64_t>(1, d.a2_oh * d.a2_ow) : m, each = d.a2_stride > 0 ? d.a2_h * d.a2_w : 1;
          if (images % units_ != 0 || !lies(s.a2, images * each * d.lda2 * es)) return false;
          uses->rows.push_back(s.a2);
          uses->shared.insert(uses->shared.end(), {s.b2, s.init2});
        }
        if (s.chained) {
          if (!share(&out->next_gemm.m, part) || !lies(s.out2, m * s.next_gemm.ldc * 2)) return false;
          uses->shared.insert(uses->shared.end(), {s.next_b, s.next_init});
          uses->results.push_back(s.out2);
          pml_hip_gemm_desc first = d;
          if (!pml_hip_gemm_chain_takes(&first, &out->next_gemm)) return false;
        }
        return tail(s, d.tail, m, uses);
      }
      case Step::Conv2d: {
        pml_hip_conv2d_desc& d = out->conv;
        const int64_t n = d.n, es = elemBytes(d.in_dtype);
        if (s.out2 >= 0 || !share(&d.n, part) || !lies(s.a, n * d.h * d.w * d.ci * es) || s.c < 0 || plan_.buffers[s.c].bytes % static_cast<size_t>(n) != 0) return false;
        if (d.init_kind && d.init_row_stride != 0) return false;
        if (PML_HIP_FLAG_MAXPOOL_OF(d.flags) && !pml_hip_conv2d_takes_maxpool(&d)) return false;
        uses->rows = {s.a};
        uses->shared = {s.b, s.init};
        uses->results = {s.c};
        return tail(s, d.tail, n * d.oh * d.ow, uses);
      }
      case Step::Dwconv2d: {
        pml_hip_dwconv2d_desc& d = out->dw;
        const int64_t n = d.n, es = elemBytes(d.dtype);
        if (s.out2 >= 0 || !share(&d.n, part) || !lies(s.a, n * d.h * d.w * d.c * es) || s.c < 0 || plan_.buffers[s.c].bytes % static_cast<size_t>(n) != 0) return false;
        uses->rows = {s.a};
        uses->shared = {s.b};
        uses->results = {s.c};
        return tail(s, d.tail, n * d.oh * d.ow, uses);
      }
      case Step::Pool2d: {
        pml_hip_pool2d_desc& d = out->pool;
        const int64_t n = d.n, es = elemBytes(d.dtype), pixels = d.oh * d.ow * d.c;
        if (!share(&d.n, part) || !lies(s.a, n * d.h * d.w * d.c * es) || !lies(s.c, n * pixels * es) || (s.out2 >= 0 && !lies(s.out2, n * pixels * 4))) return false;
        uses->rows = {s.a};
        uses->results = {s.c, s.out2};
        return s.operands.empty();
      }
      case Step::Softmax:
      case Step::Argmax:
      case Step::TopK: {
        pml_hip_softmax_desc& d = out->sm;
        const int64_t rows = d.rows, es = elemBytes(d.dtype);
        if (!share(&d.rows, part) || !lies(s.a, rows * d.cols * es)) return false;
        if (s.kind == Step::Softmax && !lies(s.c, rows * d.cols * es)) return false;
        if (s.kind == Step::Argmax && !lies(s.c, rows * 4)) return false;
        if (s.kind == Step::TopK && ((s.c >= 0 && !lies(s.c, rows * s.topk * es)) || (s.out2 >= 0 && !lies(s.out2, rows * s.topk * 4)))) return false;
        uses->rows = {s.a};
        uses->results = {s.c, s.out2};
        return s.operands.empty();
      }
      case Step::Product: {
        pml_hip_product_desc& d = out->prod;
        if (s.out2 >= 0 || s.b_off != 0) return false;
        const int64_t es = elemBytes(d.in_dtype), os = elemBytes(d.out_dtype);
        if (d.init_kind && d.init_row_stride != 0) return false;
        uses->results = {s.c};
        if (d.n_batch > 0) {
          const int64_t n = d.batch[0];
          if (!share(&d.batch[0], part) || !lies(s.c, n * d.c_batch[0] * os)) return false;
          for (const auto& [buf, stride] : {std::make_pair(s.a, d.a_batch[0]), std::make_pair(s.b, d.b_batch[0])}) {
            if (stride != 0 && !lies(buf, n * stride * es)) return false;
            (stride != 0 ? uses->rows : uses->shared).push_back(buf);
          }
        } else {
          const int64_t m = d.m;
          if (!share(&d.m, part) || !lies(s.a, m * d.a_ms * es) || !lies(s.c, m * d.c_ms * os)) return false;
          uses->rows = {s.a};
          uses->shared = {s.b};
        }
        uses->shared.push_back(s.init);
        for (size_t q = 0; q < s.operands.size(); ++q) {
          if (d.tail.operand_row_stride[q] != 0) return false;
          uses->shared.push_back(s.operands[q]);
        }
        return true;
      }
      default: return false;
    }
  }

  // A row program: its operands and results are lists.
  bool sliceRows(const Step& s, int64_t part, Step* out, Uses* uses) const {
    *out = s;
    *uses = {};
    pml_hip_rows_desc& d = out->rows;
    const int64_t rows = d.rows, es = elemBytes(d.dtype);
    if (!share(&d.rows, part) || !pml_hip_rows_takes(&d)) return false;
    std::vector<int> kind(s.operands.size(), 0), stored(s.outs.size(), 0);  // bytes a row, -1: shared
    auto note = [&](std::vector<int>* of, int index, int bytes) {
      if (index < 0 || static_cast<size_t>(index) >= of->size() || ((*of)[index] != 0 && (*of)[index] != bytes)) return false;
      (*of)[index] = bytes;
      return true;
    };
    auto operand = [&](int k, int index) {
      if (k == PML_HIP_ROWS_FULL) return note(&kind, index, static_cast<int>(d.cols * es));
      if (k == PML_HIP_ROWS_ROW) return note(&kind, index, static_cast<int>(es));
      if (k == PML_HIP_ROWS_COLUMNS || k == PML_HIP_ROWS_ONE) return note(&kind, index, -1);
      return true;
    };
    for (int i = 0; i < d.n_steps; ++i) {
      const pml_hip_rows_step& p = d.steps[i];
      if (!operand(p.a_kind, p.a) || !operand(p.b_kind, p.b)) return false;
      if (p.kind == PML_HIP_ROWS_STORE && !note(&stored, p.dst, static_cast<int>(d.cols * es))) return false;
      if (p.kind == PML_HIP_ROWS_STORE_SCALAR && !note(&stored, p.dst, static_cast<int>(es))) return false;
    }
    for (size_t i = 0; i < kind.size(); ++i) {
      if (kind[i] > 0 && !lies(s.operands[i], rows * kind[i])) return false;
      (kind[i] > 0 ? uses->rows : uses->shared).push_back(s.operands[i]);
    }
    for (size_t i = 0; i < stored.size(); ++i) {
      if (stored[i] <= 0 || !lies(s.outs[i], rows * stored[i])) return false;
      uses->results.push_back(s.outs[i]);
    }
    return true;
  }

 private:
  const Plan& plan_;
  int64_t units_;
  bool share(int64_t* extent, int64_t part) const {
    if (*extent <= 0 || *extent % units_ != 0) return false;
    *extent = *extent / units_ * part;
    return true;
  }
  bool lies(int buf, int64_t bytes) const { return buf >= 0 && bytes > 0 && plan_.buffers[buf].bytes == static_cast<size_t>(bytes); }
  bool tail(const Step& s, const pml_hip_epilogue& t, int64_t rows, Uses* uses) const {
    for (size_t q = 0; q < s.operands.size(); ++q) {
      const int64_t rs = t.operand_row_stride[q];
      if (rs != 0 && !lies(s.operands[q], rows * rs * elemBytes(t.operand_dtype[q]))) return false;
      (rs != 0 ? uses->rows : uses->shared).push_back(s.operands[q]);
    }
    return true;
  }
};

// Microseconds that a `count`-th of a step is taken to take: memory at 3.5 TB/s, matrix products at 500 TFLOP/s, and no less than a
// launch with a few memory latencies in it.
double stepUs(const Step& s, int64_t count) { return std::max(6.0, 2.0 + std::max(s.bytes / 3.5e6, s.flops / 500e6) / static_cast<double>(count)); }
constexpr double kLinkBytesPerUs = 56e3;
// What a part costs besides: its copies', waits' and launches' places in three queues (18 to 25 us between two parts' kernels)
constexpr double kPartUs = 20;
// A part has at least so many bytes to carry, up or down (75 us on the link): every operand and result of every part is a copy of its
// own.  (6 MB up and down around three launches in four parts: 465 us, 394 in one.)
constexpr int64_t kPartBytes = 4 << 20;
// Kernels fill the chip less well with a part of their work: nine steps of ResNet-50 that take 610 us on 128 images take 764 in four
// parts.  us a run with four, three and two parts: 128 images 2440, 2437, 2411, 96 images 2093, 2082, 2055, 64 images 1645, 1596,
// 1582; mean-variance normalisation of 4096x1000 fp32 597, 601, 608.
constexpr int kMostParts = 2;

}  // namespace

// What is bound by the link is cut where its kernels would wait for it: ResNet-50 on 128 images, 38 MB up ahead of the first launch,
// 2630 us a run with the kernels behind the copies, 2411 with its first steps in two parts; mean-variance normalisation of 4096x1000
// fp32, 16 MB either way, 866 and 608 to 680; of 2048x1024, 8 MB, 428 and 391.
void Planner::sliceSteps() {
  Plan& p = *plan_;
  int64_t link_in = 0, link_out = 0, units = 0, largest = 0;
  for (const auto& v : prog_->inputs) {
    const auto& sizes = v->shape.sizes;
    const int64_t bytes = static_cast<int64_t>(v->shape.getByteSize());
    link_in += bytes;
    if (!sizes.empty() && bytes > largest) {  // (the leading dimension of the largest input is what is sliced)
      largest = bytes;
      units = sizes[0];
    }
  }
  for (int b : p.output_buffers) link_out += static_cast<int64_t>(p.buffers[b].bytes);
  const int64_t slices = std::min<int64_t>({kMostParts, std::max(link_in, link_out) / kPartBytes, units});
  if (slices < 2) return;
  const int64_t part = (units + slices - 1) / slices, count = (units + part - 1) / part, last = units - (count - 1) * part;
  if (count < 2) return;

  Slicer slicer(p, units);
  const size_t nb = p.buffers.size();
  enum { Unseen, Sliced, Shared };
  std::vector<int> as(nb, Unseen);
  std::vector<int> writers(nb, 0);
  for (const Step& s : p.steps) {
    for (int w : {s.c, s.out2})
      if (w >= 0) ++writers[w];
    for (int w : s.outs) ++writers[w];
  }
  std::vector<Step> first, behind;
  int64_t carried = 0;  // bytes of the inputs that arrive in parts
  size_t n = 0;
  std::vector<int64_t> arriving;  // ... for the steps so far
  for (; n < p.steps.size(); ++n) {
    const Step& s = p.steps[n];
    Step a, b;
    Uses uses, same;
    const bool ok = s.kind == Step::Rows ? slicer.sliceRows(s, part, &a, &uses) && slicer.sliceRows(s, last, &b, &same)
                                         : slicer.slice(s, part, &a, &uses) && slicer.slice(s, last, &b, &same);
    if (!ok) break;
    bool fits = true;
    auto use = [&](int buf, int how) {
      if (buf < 0) return;
      const BufferInfo& info = p.buffers[buf];
      if (info.kind == BufferInfo::Constant) {
        fits = fits && how == Shared;
        return;
      }
      if (info.kind == BufferInfo::Input) {
        const auto& sizes = prog_->inputs[info.index]->shape.sizes;
        if (how == Sliced && (sizes.empty() || sizes[0] != units)) fits = false;
        if (as[buf] == Unseen) {
          as[buf] = how;
          if (how == Sliced) carried += static_cast<int64_t>(info.bytes);
        }
      }
      fits = fits && as[buf] == how;  // (what a slice computed is there in parts, and read in the same ones)
    };
    const std::vector<int> before = as;
    const int64_t carried_before = carried;
    for (int r : uses.rows) use(r, Sliced);
    for (int r : uses.shared) use(r, Shared);
    for (int w : uses.results) {
      if (w < 0) continue;
      if (p.buffers[w].kind == BufferInfo::Input || p.buffers[w].kind == BufferInfo::Constant || writers[w] != 1 || as[w] != Unseen) fits = false;
      as[w] = Sliced;
    }
    if (!fits) {
      as = before;
      carried = carried_before;
      break;
    }
    first.push_back(a);
    behind.push_back(b);
    arriving.push_back(carried);
  }
  // How many of them: the run's end as the link up, the kernels and the link down follow one another, part by part.
  auto ends = [&](size_t steps) {
    const double whole_up = static_cast<double>(link_in - (steps ? arriving[steps - 1] : 0)) / kLinkBytesPerUs;
    double up = whole_up, done = up, down = 0, part_us = kPartUs;
    const bool complete = steps == p.steps.size();
    for (size_t i = 0; i < steps; ++i) part_us += stepUs(p.steps[i], count);
    if (steps)
      for (int64_t k = 0; k < count; ++k) {
        up += static_cast<double>(arriving[steps - 1]) / kLinkBytesPerUs / static_cast<double>(count);
        done = std::max(up, done) + part_us;
        if (complete) down = std::max(done, down) + static_cast<double>(link_out) / kLinkBytesPerUs / static_cast<double>(count);
      }
    for (size_t i = steps; i < p.steps.size(); ++i) done += stepUs(p.steps[i], 1);
    return complete && steps ? down : done + static_cast<double>(link_out) / kLinkBytesPerUs;
  };
  const double unsliced = ends(0);
  size_t best = 0;
  for (size_t steps = 1; steps <= n; ++steps)
    if (ends(steps) < ends(best)) best = steps;
  n = best;
  if (n == 0 || arriving[n - 1] < kPartBytes || ends(n) > 0.95 * unsliced) return;
  first.resize(n);
  behind.resize(n);

  // Values that live and die among the sliced steps hold a part at a time; the others lie part behind part.
  p.slices = static_cast<int>(count);
  p.uneven = last != part;
  p.sliced = std::move(first);
  p.sliced_last = std::move(behind);
  p.part_bytes.assign(nb, 0);
  std::vector<char> inside(nb, 0), outside(nb, 0);
  auto each = [](const Step& s, auto&& fn) {
    for (int b : {s.a, s.b, s.c, s.init, s.out2, s.a2, s.b2, s.init2}) fn(b);
    for (int b : s.operands) fn(b);
    for (int b : s.outs) fn(b);
  };
  for (size_t i = 0; i < p.steps.size(); ++i)
    each(p.steps[i], [&](int b) {
      if (b >= 0) (i < n ? inside : outside)[b] = 1;
    });
  for (size_t b = 0; b < nb; ++b) {
    BufferInfo& info = p.buffers[b];
    if (!inside[b] || as[b] != Sliced) continue;
    const size_t part_bytes = info.bytes / static_cast<size_t>(units) * static_cast<size_t>(part);
    if (info.kind == BufferInfo::Temp && !outside[b])
      info.bytes = part_bytes;
    else
      p.part_bytes[b] = part_bytes;
  }
}

// A run of launches of its own costs a wait between two queues and a graph.  It begins behind a result of 4 MB and more (75 us on
// the link), which goes down beside it: 1024 x 1024 of a product ahead of two small launches 186 us a call, 163 in two runs, 4096 x
// 2048 848 and 736.  And it begins where an operand of 4 MB and more is needed first, if what lies ahead for the operand to go up
// beside takes longer than that: launches, or results that go down.  (One, two, four, six, ten small launches ahead of a product with
// 10000 x 128: 288, 284, 294, 308, 338 us a call, in two runs 316, 318, 315, 321, 335; 23 products of 17 x 128 and 128 x 370,
// softmax, 370 x 128 283 and 289.)
constexpr double kRunUs = 60;
constexpr int64_t kRunBytes = 4 << 20;

void Planner::separateRuns() {
  Plan& p = *plan_;
  std::vector<int> writer(p.buffers.size(), -1);  // the last step that writes a buffer
  for (size_t i = 0; i < p.steps.size(); ++i) {
    for (int b : {p.steps[i].c, p.steps[i].out2})
      if (b >= 0) writer[b] = static_cast<int>(i);
    for (int b : p.steps[i].outs) writer[b] = static_cast<int>(i);
  }
  std::vector<char> up(p.buffers.size(), 0);
  bool behind = false;   // a long result (or the parts of the steps before)
  double ahead = 0;      // us of the run so far: its launches, and its results' way down
  for (size_t i = 0; i < p.steps.size(); ++i) {
    const Step& s = p.steps[i];
    int64_t coming = 0, going = 0;
    auto reads = [&](int b) {
      if (b < 0 || p.buffers[b].kind != BufferInfo::Input || up[b]) return;
      up[b] = 1;
      coming += static_cast<int64_t>(p.buffers[b].bytes);
    };
    for (int b : {s.a, s.b, s.init, s.a2, s.b2, s.init2, s.next_b, s.next_init, s.out2, s.c}) reads(b);
    for (int b : s.operands) reads(b);
    if (i < p.sliced.size()) {
      behind = true;
      continue;
    }
    if (behind || (coming >= kRunBytes && ahead >= kRunUs)) {
      p.runs.push_back(i);
      ahead = 0;
    }
    for (int b : p.output_buffers)
      if (writer[b] == static_cast<int>(i)) going += static_cast<int64_t>(p.buffers[b].bytes);
    ahead += stepUs(s, 1) + static_cast<double>(going) / kLinkBytesPerUs;
    behind = going >= kRunBytes;
  }
}

}  // namespace pmlc::target::hip
