// The other layer entry points: convolution (implicit GEMM, filter stamps, generator windows), the ReLU step's
// C entry points and the layer loop of NN.reach in one call.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>

#include "internal.h"

using namespace nnvhip;

static const ColBox kAnyBox = {0, 0, 0, 0};  // stands for a window table in a question about sizes

extern "C" {

int nnvhip_affine_conv2d(nnvhip_ctx* c, const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t count,
                         nnvhip_star* const* in, nnvhip_star** out) {
  CHECK_CTX(c);
  // (what the caller knows about the layers behind is for this call, whatever becomes of it)
  const nnvhip_conv2d* const behind_conv = c->behind_conv;
  const nnvhip_fc* const behind_fc = c->behind_fc;
  c->behind_conv = nullptr;
  c->behind_fc = nullptr;
  if (!cv || cv->ctx != c) NNV_FAIL(NNVHIP_ERR_ARG, "invalid layer handle");
  NNV_TRY(check_set_array(c, count, in, out));
  if (H <= 0 || W <= 0) NNV_FAIL(NNVHIP_ERR_SHAPE, "The input is not an ImageStar object");
  for (int64_t i = 0; i < count; ++i) {
    if (in[i]->N % (H * W) != 0) NNV_FAIL(NNVHIP_ERR_SHAPE, "Inconsistent dimension in the ImageStar and the original Star set");
    int64_t ch = in[i]->N / (H * W);
    if (ch != cv->Cin)
      NNV_FAIL(NNVHIP_ERR_SHAPE, "Input set contains %lld channels while the convolutional layers has %lld channels",
               (long long)ch, (long long)cv->Cin);
  }
  int64_t Ho = 0, Wo = 0;
  NNV_TRY(nnvhip_conv2d_output_size(cv, H, W, &Ho, &Wo));
  int64_t Nout = Ho * Wo * cv->Cout;
  if (Nout >= (int64_t(1) << 31) || in[0]->N >= (int64_t(1) << 31)) NNV_FAIL(NNVHIP_ERR_SHAPE, "image too large");
  std::vector<nnvhip_star*> outs;
  bool contig = false;
  int64_t cols = 0;
  NNV_TRY(c->begin_op());
  int st = make_affine_outputs(c, count, in, Nout, &outs, &contig, &cols);
  // generator images that are scaled unit vectors (box ImageStars, columns appended by a ReLU) turn
  // into stamps of the filter; the implicit GEMM runs over the leading dense images only
  std::vector<ConvStampSet> stamps((size_t)count);
  auto mask_on_load = [&](const nnvhip_star* s) {
    return !c->no_conv_mask && s->cls != nullptr && conv2d_can_mask(cv, H, W, Ho, Wo, s->ld);
  };
  bool any_stamps = false;
  int64_t max_m = 0;
  // Windows of the generator images (internal.h, nnvhip_star::box).  The output's come from the input's windows and
  // from the pixels of its unit-vector columns (without either an image counts as full); where the input's dense
  // images have small windows the implicit GEMM computes inside the output windows only.
  const bool track_boxes = !c->no_conv_boxes && H < 32768 && W < 32768 && Ho < 32768 && Wo < 32768;
  struct Plan {
    int64_t nc = 0, dense = 0, m = 0;
    bool in_ok = false;      // the input's windows describe its dense images
    bool out_boxes = false;  // the output gets windows
    bool compact = false;    // the dense images are computed inside their windows only
    int dense_eh = 0, dense_ew = 0;
  };
  std::vector<Plan> plan((size_t)count);
  for (int64_t i = 0; i < count; ++i) {
    Plan& pl = plan[i];
    pl.nc = in[i]->n + 1;
    pl.dense = (!c->dense_affine && in[i]->oh_from > 0 && in[i]->oh_from < pl.nc) ? in[i]->oh_from : pl.nc;
    pl.m = pl.nc - pl.dense;
    if (!track_boxes) continue;
    pl.in_ok = in[i]->box != nullptr && in[i]->box_H == H && in[i]->box_W == W && in[i]->box_cols >= pl.dense;
    pl.out_boxes = pl.in_ok || (pl.m > 0 && pl.dense == 1);
    if (pl.in_ok && pl.dense > 1) {
      pl.dense_eh = (int)conv_box_extent(cv, 0, in[i]->box_eh, Ho);
      pl.dense_ew = (int)conv_box_extent(cv, 1, in[i]->box_ew, Wo);
      // (any table will do for the question; the real one is made below)
      pl.compact = conv2d_in_windows(cv, H, W, Ho, Wo, in[i]->ld, pl.dense, in[i]->box, pl.dense_eh, pl.dense_ew);
    }
  }
  // Images with windows go by output position (conv_window.hip), which leaves their range sums too; not when the caller
  // wants every column in memory (the zeros around the windows are then written first).
  auto by_position = [&](const Plan& pl) {
    return !c->eager_cols && pl.out_boxes && pl.compact && conv_window_takes(cv, H, W, Ho, Wo, pl.dense, pl.dense_eh, pl.dense_ew);
  };
  {
    // The implicit GEMM reads whole images: pending row resets are run first, and sets whose unit-vector
    // columns take part in the contraction get those written out.  (A pending reset alone is applied by the
    // kernel as it loads, from one bit per row, where that fits; images that are in memory inside their windows
    // only are fine for the kernel that stays inside the windows.)
    // Images kept pixel by pixel are for the kernel that goes by output position; another one gets their columns first.
    std::vector<nnvhip_star*> full, prefix, columns;
    for (int64_t i = 0; i < count; ++i) {
      const ColSource& cs = in[i]->cs;
      if (cs.in_pixels() && !(by_position(plan[i]) && conv_window_takes_pixels(cv, H, W, cs.pix_eh, cs.pix_ew))) columns.push_back(in[i]);
    }
    if (st == NNVHIP_OK && !columns.empty()) st = write_pending_columns(c, (int64_t)columns.size(), columns.data());
    for (int64_t i = 0; i < count; ++i) {
      const ColSource& cs = in[i]->cs;
      if (plan[i].dense > in[i]->stored_cols())
        full.push_back(in[i]);
      else if (cs.pending || cs.zero_to > 1 || cs.delta_pending() || (cs.win_pending() && !plan[i].compact) ||
               (in[i]->rows_pending && !mask_on_load(in[i])))
        prefix.push_back(in[i]);
    }
    if (st == NNVHIP_OK && !full.empty()) st = ensure_dense_batch(c, (int64_t)full.size(), full.data());
    if (st == NNVHIP_OK && !prefix.empty()) st = ensure_dense_batch(c, (int64_t)prefix.size(), prefix.data(), false);
  }
  // range sums of the stamped columns, left on the output handles: one buffer for the call
  for (int64_t i = 0; i < count; ++i) {
    any_stamps = any_stamps || plan[i].m > 0;
    max_m = std::max<int64_t>(max_m, plan[i].m);
  }
  const int64_t sch = any_stamps && st == NNVHIP_OK ? conv_stamp_chunks(cv, outs[0]->ld, count, max_m) : 0;
  std::vector<int64_t> parts((size_t)count, 0), chunk_at((size_t)count + 1, 0);  // parts > 0: by position
  for (int64_t i = 0; i < count; ++i) {
    const Plan& pl = plan[i];
    if (by_position(pl))
      parts[(size_t)i] = conv_window_parts(cv, Ho, Wo, pl.dense, pl.dense_eh, pl.dense_ew);
    chunk_at[(size_t)i + 1] = chunk_at[(size_t)i] + parts[(size_t)i] + sch;
  }
  BufRef sums;
  if (chunk_at[(size_t)count] > 0 && st == NNVHIP_OK) st = c->alloc(sizeof(double) * 4 * outs[0]->ld * chunk_at[(size_t)count], &sums);
  // Bound on the windows of a set's output columns.
  auto out_extent = [&](const Plan& pl, int64_t* eh, int64_t* ew) {
    *eh = pl.dense > 1 ? pl.dense_eh : 0;
    *ew = pl.dense > 1 ? pl.dense_ew : 0;
    if (pl.m > 0) {
      *eh = std::max(*eh, conv_box_extent(cv, 0, 1, Ho));
      *ew = std::max(*ew, conv_box_extent(cv, 1, 1, Wo));
    }
  };
  // The output's images are kept pixel by pixel (ColSource::pix) where every one of them is made by a kernel that can write
  // them so, and the layer behind the next ReLU step is known and will read them so: another reader would have the columns
  // written first, which costs what is saved here.
  auto can_write_pixels = [&](int64_t i) {
    const Plan& pl = plan[(size_t)i];
    if ((behind_conv == nullptr && behind_fc == nullptr) || c->eager_cols || c->eager_rows || c->eager_tail || c->dense_affine) return false;
    if (!pl.out_boxes || pl.nc < 2 || (pl.dense > 1 && parts[(size_t)i] == 0) || (pl.m > 0 && !(conv_stamps_by_pixel(cv) && cv->K <= 1024)) || cv->Wk == nullptr)
      return false;
    int64_t eh = 0, ew = 0;
    out_extent(pl, &eh, &ew);
    return eh >= 1 && ew >= 1;
  };
  auto conv_reads_pixels = [&](int64_t i) {  // (which goes set by set)
    const Plan& pl = plan[(size_t)i];
    int64_t eh = 0, ew = 0, H2 = 0, W2 = 0;
    out_extent(pl, &eh, &ew);
    const int64_t ldo = round_up(Nout, kLdAlign);
    if (behind_conv->ctx != c || behind_conv->Cin != cv->Cout || c->no_conv_mask || nnvhip_conv2d_output_size(behind_conv, Ho, Wo, &H2, &W2) != NNVHIP_OK)
      return false;
    const int eh2 = (int)conv_box_extent(behind_conv, 0, eh, H2), ew2 = (int)conv_box_extent(behind_conv, 1, ew, W2);
    return conv2d_can_mask(behind_conv, Ho, Wo, H2, W2, ldo) &&
           conv2d_in_windows(behind_conv, Ho, Wo, H2, W2, ldo, pl.nc, &kAnyBox, eh2, ew2) &&
           conv_window_takes(behind_conv, Ho, Wo, H2, W2, pl.nc, eh2, ew2) && conv_window_takes_pixels(behind_conv, Ho, Wo, eh, ew);
  };
  auto fc_reads_pixels = [&] {  // (which takes all sets of an array that way or none)
    if (behind_fc->ctx != c || behind_fc->K != Nout || !fc_window_takes(behind_fc, Ho, Wo)) return false;
    int64_t eh0 = 0, ew0 = 0, images = 0;
    for (int64_t i = 0; i < count; ++i) {
      if (!can_write_pixels(i)) return false;
      int64_t eh = 0, ew = 0;
      out_extent(plan[(size_t)i], &eh, &ew);
      if (i == 0) eh0 = eh, ew0 = ew;
      const int64_t nc = plan[(size_t)i].nc;
      if (eh != eh0 || ew != ew0 || nc > kFcWindowColumns || (double)behind_fc->Mp * (double)behind_fc->Kp * (double)nc * (double)count < 4.0e6) return false;
      images += nc - 1;
    }
    return fc_window_tile_of(behind_fc, count, images, Ho, Wo, eh0, ew0) > 0;
  };
  const bool for_fc = behind_fc != nullptr && st == NNVHIP_OK && fc_reads_pixels();
  auto keep_pixels = [&](int64_t i) { return behind_conv != nullptr ? can_write_pixels(i) && conv_reads_pixels(i) : for_fc; };
  std::vector<int64_t> pix_at((size_t)count, -1);
  BufRef pixels;
  {
    int64_t total = 0;
    for (int64_t i = 0; i < count && st == NNVHIP_OK; ++i) {
      if (!keep_pixels(i)) continue;
      int64_t eh = 0, ew = 0;
      out_extent(plan[(size_t)i], &eh, &ew);
      pix_at[(size_t)i] = total;
      total += plan[(size_t)i].nc * round_up(eh * ew * cv->Cout, kLdAlign);  // (column 0, the centre, stays in the matrix)
    }
    // (the buffer comes on top of the matrices: without room for it they hold the columns)
    const bool kept = total > 0 && c->pixel_bytes + 8 * total <= c->pixel_limit && c->alloc(sizeof(double) * total, &pixels, true) == NNVHIP_OK;
    if (kept) {
      pixels->tally = &c->pixel_bytes;
      c->pixel_bytes += (int64_t)pixels->bytes;
    } else {
      std::fill(pix_at.begin(), pix_at.end(), -1);
    }
    if (kept && c->poison_pending) NNV_HIP_TRY(hipMemsetAsync(pixels->ptr, 0xff, sizeof(double) * total, c->stream));
  }
  // windows of the output's columns and the pixel tables of the unit-vector columns: one buffer each, one launch
  std::vector<ConvSetup> setup((size_t)count);
  BufRef boxes, invs, orders;
  int64_t box_cols = 0, inv_sets = 0, order_ints = 0;
  const int64_t first_stride = round_up(Ho * Wo + 1, kLdAlign);
  const int64_t inv_stride = round_up(in[0]->N, kLdAlign);
  auto wants_inv = [&](int64_t i) { return plan[i].m > 0 && in[i]->oh_inv == nullptr && conv_stamps_by_pixel(cv); };
  for (int64_t i = 0; i < count; ++i) {
    if (plan[i].out_boxes) box_cols += plan[i].nc;
    if (wants_inv(i)) ++inv_sets;
    if (parts[(size_t)i] > 0) order_ints += first_stride + plan[i].dense;
  }
  if (st == NNVHIP_OK && order_ints > 0) st = c->alloc(sizeof(int32_t) * (size_t)order_ints, &orders);
  if (st == NNVHIP_OK && box_cols > 0) st = c->alloc(sizeof(ColBox) * (size_t)box_cols, &boxes);
  if (st == NNVHIP_OK && inv_sets > 0) st = c->alloc(sizeof(int32_t) * (size_t)(inv_stride * inv_sets), &invs);
  if (st == NNVHIP_OK && (box_cols > 0 || inv_sets > 0)) {
    int64_t box_at = 0, inv_at = 0, order_at = 0;
    for (int64_t i = 0; i < count; ++i) {
      const Plan& pl = plan[i];
      ConvSetup& su = setup[(size_t)i];
      su = ConvSetup{pl.in_ok ? in[i]->box : nullptr, in[i]->oh_idx, nullptr, nullptr, (int32_t)pl.dense, (int32_t)pl.m, (int32_t)in[i]->N, nullptr,
                     nullptr};
      if (pl.out_boxes) {
        su.out_box = boxes->as<ColBox>() + box_at;
        box_at += pl.nc;
      }
      if (wants_inv(i)) {
        su.inv = invs->as<int32_t>() + inv_at;
        inv_at += inv_stride;
      }
      if (parts[(size_t)i] > 0) {
        su.first = orders->as<int32_t>() + order_at;
        su.order = su.first + first_stride;
        order_at += first_stride + pl.dense;
      }
    }
    st = launch_conv_setup(c, cv, H, W, Ho, Wo, count, setup.data());
    for (int64_t i = 0; i < count && st == NNVHIP_OK; ++i)
      if (setup[(size_t)i].inv != nullptr) {  // (kept on the input: its columns do not change, and an input set is usually mapped again)
        in[i]->oh_inv_buf = invs;
        in[i]->oh_inv = setup[(size_t)i].inv;
      }
  }
  std::vector<ConvJob> jobs;
  std::vector<int64_t> job_of;
  std::vector<ConvWindowSet> windows;
  std::vector<char> stamped((size_t)count, 0);  // sets whose stamps go into another launch
  jobs.reserve((size_t)count);
  for (int64_t i = 0; i < count && st == NNVHIP_OK; ++i) {
    const Plan& pl = plan[i];
    nnvhip_star* o = outs[i];
    const ColBox* ob = nullptr;
    if (pl.out_boxes) {
      int64_t eh = 0, ew = 0;
      out_extent(pl, &eh, &ew);
      ob = setup[(size_t)i].out_box;
      o->box_buf = boxes;
      o->box = ob;
      o->box_cols = pl.nc;
      o->box_H = (int32_t)Ho;
      o->box_W = (int32_t)Wo;
      o->box_eh = (int32_t)eh;
      o->box_ew = (int32_t)ew;
    }
    // Images with windows are written inside them only; the zeros around them wait for a reader of whole
    // columns (ColSource::win_*).  Not when the caller wants every column in memory.
    const bool lazy = ob != nullptr && !c->eager_cols;
    const int64_t win_from = lazy ? (pl.compact ? 1 : pl.dense) : 0;
    const int64_t win_to = lazy ? (pl.m > 0 ? pl.nc : (pl.compact ? pl.dense : 0)) : 0;
    if (win_to > win_from) {
      o->cs.win_box_buf = o->box_buf;
      o->cs.win_box = ob;
      o->cs.win_from = win_from;
      o->cs.win_to = win_to;
      o->cs.win_rows = Nout;
      o->cs.win_H = (int32_t)Ho;
      o->cs.win_W = (int32_t)Wo;
      if (c->poison_pending)  // debugging aid: NaNs where nothing will be written
        NNV_HIP_TRY(hipMemsetAsync(o->V + win_from * o->ld, 0xff, sizeof(double) * o->ld * (win_to - win_from), c->stream));
    }
    stamps[i].idx = in[i]->oh_idx;
    stamps[i].scale = in[i]->oh_scale;
    stamps[i].out = o->V + pl.dense * o->ld;
    stamps[i].plb = o->plb + (pl.dense - 1);
    stamps[i].pub = o->pub + (pl.dense - 1);
    stamps[i].part = sums ? sums->as<double>() + 4 * outs[0]->ld * (chunk_at[(size_t)i] + parts[(size_t)i]) : nullptr;
    stamps[i].m = (int32_t)pl.m;
    stamps[i].pixel_col = in[i]->oh_inv;
    stamps[i].win_only = (lazy && pl.m > 0) ? 1 : 0;
    stamps[i].pix = nullptr;
    if (pix_at[(size_t)i] >= 0) {
      o->cs.pix_buf = pixels;
      o->cs.pix = pixels->as<double>() + pix_at[(size_t)i];
      o->cs.pix_ld = round_up((int64_t)o->box_eh * o->box_ew * cv->Cout, kLdAlign);
      o->cs.pix_eh = o->box_eh;
      o->cs.pix_ew = o->box_ew;
      ++c->routes[NNVHIP_ROUTE_CONV_PIXELS];
      if (pl.m > 0) {
        stamps[i].pix = pixels->as<double>() + pix_at[(size_t)i] + pl.dense * o->cs.pix_ld;
        stamps[i].pix_ld = o->cs.pix_ld;
        stamps[i].pix_eh = o->box_eh;
        stamps[i].pix_ew = o->box_ew;
      }
    }
    if (parts[(size_t)i] > 0) {
      const bool stamp = sch == 1 && pl.m > 0 && in[i]->oh_inv != nullptr && conv_stamps_by_pixel(cv);
      windows.push_back(ConvWindowSet{in[i], o, pl.dense, pl.dense_eh, pl.dense_ew, setup[(size_t)i].order, setup[(size_t)i].first, parts[(size_t)i],
                                      sums->as<double>() + 4 * o->ld * chunk_at[(size_t)i], stamp ? &stamps[i] : nullptr});
      if (stamp) stamped[(size_t)i] = 1;
    } else {
      job_of.push_back(i);
      jobs.push_back(ConvJob{in[i]->V, in[i]->ld, o->V, pl.dense, in[i]->rows_pending ? in[i]->cls : nullptr,
                             in[i]->rows_pending ? in[i]->keep_bits : nullptr, pl.compact ? ob : nullptr, pl.dense_eh, pl.dense_ew,
                             pl.compact ? in[i]->box : nullptr, pl.compact && lazy, sch == 1 ? &stamps[i] : nullptr, false});
    }
  }
  if (st == NNVHIP_OK) st = launch_conv2d(c, cv, H, W, Ho, Wo, outs[0]->ld, jobs);
  for (size_t k = 0; k < jobs.size(); ++k) stamped[(size_t)job_of[k]] = jobs[k].stamped ? 1 : 0;
  if (st == NNVHIP_OK)
    st = launch_conv_window(c, cv, H, W, Ho, Wo, outs[0]->ld, (int64_t)windows.size(), windows.data());
  if (st == NNVHIP_OK && any_stamps) {
    // the stamp pass also leaves the range sums of its columns on the output handles; sets whose stamps went into
    // their convolution's launch are done
    std::vector<ConvStampSet> rest = stamps;
    bool any_left = false;
    for (int64_t i = 0; i < count; ++i) {
      if (stamped[(size_t)i]) rest[(size_t)i].m = 0;
      any_left = any_left || rest[(size_t)i].m > 0;
    }
    if (any_left) st = launch_conv_stamps(c, cv, H, W, Ho, Wo, outs[0]->ld, count, rest.data(), sch);
    for (int64_t i = 0; i < count && st == NNVHIP_OK; ++i)
      if (stamps[i].m > 0) {
        outs[i]->rng_buf = sums;
        outs[i]->rng_part = stamps[i].part;
        outs[i]->rng_chunks = sch;
        outs[i]->rng_first_col = (in[i]->n + 1) - stamps[i].m;
      }
  }
  for (int64_t i = 0; i < count && st == NNVHIP_OK; ++i) {  // ... and with the images' own, every column has its sums
    if (parts[(size_t)i] == 0) continue;
    outs[i]->rng_buf = sums;
    outs[i]->rng_part = sums->as<double>() + 4 * outs[0]->ld * chunk_at[(size_t)i];
    outs[i]->rng_chunks = parts[(size_t)i] + (stamps[i].m > 0 ? sch : 0);
    outs[i]->rng_first_col = 1;
  }
  // padding rows of every column of the call (they lie back to back)
  if (st == NNVHIP_OK) st = launch_zero_pad_rows(c, outs[0]->V, outs[0]->ld, Nout, cols);
  if (st == NNVHIP_OK) st = c->end_op();
  if (st != NNVHIP_OK) {
    release_all(outs);
    return st;
  }
  for (int64_t i = 0; i < count; ++i) out[i] = outs[i];
  return NNVHIP_OK;
}

int nnvhip_relu_relax(nnvhip_ctx* c, int order, double relax_factor, int64_t count, nnvhip_star* const* in,
                      nnvhip_star** out) {
  CHECK_CTX(c);
  NNV_TRY(check_set_array(c, count, in, out));
  if (order != NNVHIP_ORDER_INDEX && order != NNVHIP_ORDER_AREA && order != NNVHIP_ORDER_RANGE)
    NNV_FAIL(NNVHIP_ERR_METHOD, "This reachability method does not exist");
  if (!(relax_factor >= 0.0 && relax_factor <= 1.0)) NNV_FAIL(NNVHIP_ERR_RELAX_FACTOR, "Invalid relax factor");
  if (relax_factor != 1.0)
    NNV_FAIL(NNVHIP_ERR_RELAX_FACTOR, "relaxFactor < 1 needs the LP-based range optimisation, which this library does not provide");
  for (int64_t i = 0; i < count; ++i)
    if (in[i]->N != in[0]->N) NNV_FAIL(NNVHIP_ERR_SHAPE, "sets of one array must have the same dimension");
  NNV_TRY(c->begin_op());
  NNV_TRY(relu_relax(c, order, count, in, out));
  return c->end_op();
}

int nnvhip_reach_is_one_launch(nnvhip_ctx* c, int64_t n_layers, const int32_t* kind, const void* const* layer, int order, int64_t count,
                               nnvhip_star* const* in, int32_t* yes) {
  if (!c) NNV_FAIL(NNVHIP_ERR_ARG, "null context");
  if (n_layers < 1 || count <= 0 || !in || !kind || !layer || !yes) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  *yes = small_chain_takes(c, n_layers, kind, layer, order, count, in) ? 1 : 0;
  return NNVHIP_OK;
}

// The layer loop of nnvhip_reach_layers.  pixels: a convolution may keep its images pixel by pixel where the layers behind it read them so.
static int layer_by_layer(nnvhip_ctx* c, int64_t n_layers, const int32_t* kind, const void* const* layer, const int64_t* hw, int order,
                          double relax_factor, int64_t count, nnvhip_star* const* in, nnvhip_star** out, bool pixels) {
  nnvhip_star* const* cur = in;
  int st = NNVHIP_OK;
  int64_t done = 0;
  for (int64_t l = 0; l < n_layers && st == NNVHIP_OK; ++l) {
    nnvhip_star** dst = out + l * count;
    // the set that is handed back is written in full by the layer that produces it
    const bool eager = l == n_layers - 1 && !c->eager_cols;
    if (eager) c->eager_cols = true;
    // (a convolution at the end writes every column and does not go by position: it reads columns)
    const bool known = pixels && kind[l] == NNVHIP_LAYER_CONV2D && l + 2 < n_layers && kind[l + 1] == NNVHIP_LAYER_RELU &&
                       !(kind[l + 2] == NNVHIP_LAYER_CONV2D && l + 2 == n_layers - 1);
    c->behind_conv = known && kind[l + 2] == NNVHIP_LAYER_CONV2D ? static_cast<const nnvhip_conv2d*>(layer[l + 2]) : nullptr;
    c->behind_fc = known && kind[l + 2] == NNVHIP_LAYER_FC ? static_cast<const nnvhip_fc*>(layer[l + 2]) : nullptr;
    switch (kind[l]) {
      case NNVHIP_LAYER_FC:
        st = nnvhip_affine_fc(c, static_cast<const nnvhip_fc*>(layer[l]), count, cur, dst);
        break;
      case NNVHIP_LAYER_CONV2D:
        if (!hw) {
          set_error("null argument");
          st = NNVHIP_ERR_ARG;
        } else {
          st = nnvhip_affine_conv2d(c, static_cast<const nnvhip_conv2d*>(layer[l]), hw[2 * l], hw[2 * l + 1], count, cur, dst);
        }
        break;
      case NNVHIP_LAYER_RELU:
        st = nnvhip_relu_relax(c, order, relax_factor, count, cur, dst);
        break;
      default:
        set_error("unknown layer kind %d", (int)kind[l]);
        st = NNVHIP_ERR_ARG;
    }
    if (eager) c->eager_cols = false;
    c->behind_conv = nullptr;
    c->behind_fc = nullptr;
    if (st == NNVHIP_OK) {
      cur = dst;
      done = l + 1;
    }
  }
  if (st != NNVHIP_OK) {
    for (int64_t t = 0; t < done * count; ++t) {
      nnvhip_star_release(out[t]);
      out[t] = nullptr;
    }
  }
  return st;
}

int nnvhip_reach_layers(nnvhip_ctx* c, int64_t n_layers, const int32_t* kind, const void* const* layer, const int64_t* hw,
                        int order, double relax_factor, int64_t count, nnvhip_star* const* in, nnvhip_star** out) {
  if (!c) NNV_FAIL(NNVHIP_ERR_ARG, "null context");
  if (n_layers < 0 || count <= 0 || !in || (n_layers > 0 && (!kind || !layer || !out))) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  int st = NNVHIP_OK;
  if (n_layers > 0 && relax_factor == 1.0) {
    // small fully connected networks: the whole loop below as one launch
    NNV_TRY(nnvhip::enter_ctx(c));
    bool taken = false;
    for (int64_t t = 0; t < n_layers * count; ++t) out[t] = nullptr;
    st = reach_small_chain(c, n_layers, kind, layer, order, count, in, out, &taken);
    if (taken) {
      if (st != NNVHIP_OK)
        for (int64_t t = 0; t < n_layers * count; ++t) {
          nnvhip_star_release(out[t]);
          out[t] = nullptr;
        }
      return st;
    }
  }
  const int64_t pixels = c->routes[NNVHIP_ROUTE_CONV_PIXELS];
  st = layer_by_layer(c, n_layers, kind, layer, hw, order, relax_factor, count, in, out, !c->no_conv_pixels);
  if (st == NNVHIP_ERR_OOM && c->routes[NNVHIP_ROUTE_CONV_PIXELS] > pixels) {
    // what its own images took on top of their matrices may be what was missing: the reach starts over with columns, and so does
    // every later one of this context
    c->pixel_limit = 0;
    st = layer_by_layer(c, n_layers, kind, layer, hw, order, relax_factor, count, in, out, false);
  }
  return st;
}

int nnvhip_relu_apply_lists(nnvhip_ctx* c, nnvhip_star* in, int64_t n_reset, const int32_t* reset_rows, int64_t m,
                            const int32_t* index, const double* lb, const double* ub, nnvhip_star** out) {
  CHECK_CTX(c);
  if (!in || in->ctx != c || !out) NNV_FAIL(NNVHIP_ERR_ARG, "invalid set handle");
  if (n_reset < 0 || m < 0 || (n_reset > 0 && !reset_rows) || (m > 0 && (!index || !lb || !ub)))
    NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  const int64_t N = in->N;
  // per-row bounds that make the classification reproduce the two lists: a reset row looks inactive
  // (ub = 0), a listed neuron carries its own (lb, ub), every other row looks active; the keys put the
  // new predicates in the order of the list
  std::vector<double> rows((size_t)(3 * N));
  double* L = rows.data();
  double* U = L + N;
  double* K = U + N;
  std::vector<char> seen((size_t)N, 0);
  for (int64_t r = 0; r < N; ++r) {
    L[r] = 0.0;
    U[r] = 1.0;
    K[r] = 0.0;
  }
  for (int64_t t = 0; t < n_reset; ++t) {
    const int64_t r = reset_rows[t];
    if (r < 0 || r >= N) NNV_FAIL(NNVHIP_ERR_ARG, "Invalid index");
    if (seen[r]) NNV_FAIL(NNVHIP_ERR_ARG, "row %lld is listed twice", (long long)r);
    seen[r] = 1;
    L[r] = -1.0;
    U[r] = 0.0;
  }
  for (int64_t t = 0; t < m; ++t) {
    const int64_t r = index[t];
    if (r < 0 || r >= N) NNV_FAIL(NNVHIP_ERR_ARG, "Invalid index");
    if (seen[r]) NNV_FAIL(NNVHIP_ERR_ARG, "row %lld is listed twice", (long long)r);
    if (!(lb[t] < 0.0 && ub[t] > 0.0)) NNV_FAIL(NNVHIP_ERR_ARG, "neuron %lld: the triangle relaxation needs lb < 0 < ub", (long long)r);
    seen[r] = 1;
    L[r] = lb[t];
    U[r] = ub[t];
    K[r] = (double)(m - t);
  }
  NNV_TRY(c->begin_op());
  BufRef dev;
  NNV_TRY(c->upload(rows.data(), sizeof(double) * 3 * N, &dev));
  ReluGiven g{dev->as<double>(), dev->as<double>() + N, dev->as<double>() + 2 * N};
  NNV_TRY(relu_relax(c, kOrderGiven, 1, &in, out, &g));
  return c->end_op();
}

}  // extern "C"
