// The batched phase kernels' host sequence (Batch, declared in batch_api.hpp). A translation
// unit of its own, compiled with the kernel arguments preloaded into SGPRs (the projections'
// first loads then wait for no argument load; the single-stream fused kernel, in runtime.hip,
// is faster without).
#include "batch_api.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

namespace stamd {

Batch::Batch(const st_config& config, bool mixed, const st_tensor* tensors, size_t count, int streams,
             int weight_dtype)
    : c_(config) {
  validate_config(c_);
  if (streams < 1 || streams > kBatchMax)
    throw Error(ST_ERR_INVALID, "Streams must be between 1 and " + std::to_string(kBatchMax));
  if (weight_dtype != ST_WEIGHTS_AS_MODEL && weight_dtype != ST_WEIGHTS_BF16)
    throw Error(ST_ERR_INVALID, "Unknown weight storage");
  if (c_.width % kBatchTile || (2 * c_.ffn) % kBatchTile)
    throw Error(ST_ERR_INVALID, "Batched streams need width and 2*ffn to be multiples of 16");
  if (mixed && weight_dtype == ST_WEIGHTS_BF16)
    throw Error(ST_ERR_INVALID, "bfloat16 weight storage applies to FP32 checkpoints only");
  prec_ = mixed ? kMixed : weight_dtype == ST_WEIGHTS_BF16 ? kBf16w : kFp32;
  streams_ = streams;
  // Padded batch: 16 or 32 rows, else a multiple of 64, so that a projection's batch groups (1 or 4
  // tiles of 16) divide it.
  streams_p_ = streams <= 16 ? 16 : streams <= 32 ? 32 : (streams + 63) / 64 * 64;
  dim_ = c_.width / c_.heads;
  if (dim_ % 4) throw Error(ST_ERR_INVALID, "Batched streams need a head dimension that is a multiple of 4");
  int device = 0;
  HIP_CHECK(hipGetDevice(&device));
  hipDeviceProp_t prop;
  HIP_CHECK(hipGetDeviceProperties(&prop, device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    throw Error(ST_ERR_DEVICE, std::string("Supported target is gfx950; found ") + prop.gcnArchName);
  stream_.create();

  // Weight arena: the single-stream runtime's (rows padded to 1 KiB slabs), with the
  // projection matrices in MFMA operand order (tiled).
  const int slab = 1024 / (prec_ == kFp32 ? 4 : 2);
  offsets_.width_p = round_up(c_.width, slab);
  offsets_.ffn_p = round_up(c_.ffn, slab);
  offsets_.features_p = round_up(c_.features, slab);
  build_arena(c_, prec_, tensors, count, offsets_, weights_, true);

  BatchArgs& a = args_;
  a.streams = streams_;
  a.streams_p = streams_p_;
  a.layers = c_.layers;
  a.width = c_.width;
  a.heads = c_.heads;
  a.dim = dim_;
  a.ffn = c_.ffn;
  a.window = c_.window;
  a.features = c_.features;
  a.width_p = offsets_.width_p;
  a.ffn_p = offsets_.ffn_p;
  a.features_p = offsets_.features_p;
  a.epsilon = c_.epsilon;
  a.weights = offsets_.weights;
  a.w_input = offsets_.w_input;
  a.w_final_norm = offsets_.w_final_norm;
  a.w_score = offsets_.w_score;
  for (int l = 0; l < c_.layers; l++) a.layer[l] = offsets_.layer[l];

  std::vector<float> freq(dim_ / 2);
  for (int j = 0; j < dim_ / 2; j++) freq[j] = std::pow(10000.0f, -(float)(2 * j) / (float)dim_);
  rope_.alloc(freq.size() * 4);
  HIP_CHECK(hipMemcpy(rope_.ptr, freq.data(), freq.size() * 4, hipMemcpyHostToDevice));
  a.rope_freq = reinterpret_cast<const float*>(rope_.ptr);

  auto zeroed = [&](DeviceBuffer& buf, size_t floats) {
    buf.alloc(floats * 4);
    HIP_CHECK(hipMemset(buf.ptr, 0, std::max<size_t>(floats * 4, 256)));
    return reinterpret_cast<float*>(buf.ptr);
  };
  // K/V rings [L][B][H][W][dh]: FP32, or FP16 in mixed mode.
  block_words_ = (size_t)c_.width * c_.window * (prec_ == kMixed ? 2 : 4) / 4;
  a.keys = zeroed(keys_, (size_t)c_.layers * streams_ * block_words_);
  a.values = zeroed(values_, (size_t)c_.layers * streams_ * block_words_);
  a.hidden = zeroed(hidden_, (size_t)streams_ * c_.layers * c_.width);
  position_.alloc((size_t)streams_ * 8);
  HIP_CHECK(hipMemset(position_.ptr, 0, (size_t)streams_ * 8));
  a.position = reinterpret_cast<unsigned long long*>(position_.ptr);
  a.in = zeroed(in_, (size_t)streams_p_ * a.features_p);
  a.x = zeroed(x_, kSquares + (size_t)streams_p_ * a.width_p) + kSquares;
  a.xn = zeroed(xn_, (size_t)streams_p_ * a.width_p);
  a.attn = zeroed(attn_, (size_t)streams_p_ * a.width_p);
  a.act = zeroed(act_, (size_t)streams_p_ * a.ffn_p);
  a.q = zeroed(q_, (size_t)streams_p_ * a.width);
  host_out_.alloc((size_t)streams_ * 4);
  a.score = reinterpret_cast<float*>(host_out_.dev);
  if (attn_split()) {
    const int row = 64 * (dim_ > 64 ? 2 : 1) + 2;
    attn_part_.alloc((size_t)streams_ * c_.heads * attn_chunks() * row * 4);
    zeroed(attn_count_, (size_t)streams_ * c_.heads);
  }
  a.rope = reinterpret_cast<float2*>(zeroed(step_rope_, (size_t)streams_p_ * dim_));
  a.slot = reinterpret_cast<int*>(zeroed(step_slot_, (size_t)streams_p_));
  host_in_.alloc((size_t)streams_ * c_.features * 4);

  args_dev_.alloc(sizeof(BatchArgs));
  HIP_CHECK(hipMemcpy(args_dev_.ptr, &args_, sizeof(BatchArgs), hipMemcpyHostToDevice));
  dargs_ = reinterpret_cast<const BatchArgs*>(args_dev_.ptr);

  // Warm up outside capture, restore the initial state, then capture the step sequence.
  launch();
  sync();
  reset(-1);
  HIP_CHECK(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
  launch();
  HIP_CHECK(hipStreamEndCapture(stream_, &graph_.g));
  graph_exec_.instantiate(graph_);
}

Batch::~Batch() {
  if (stream_) (void)hipStreamSynchronize(stream_);  // before the buffers are freed
}

// Column tiles of a projection's workgroup with one batch tile (project).
int Batch::column_tiles(int cols) const {
  const int batch_tiles = streams_p_ / kBatchTile;
  for (int ct = 4; ct > 1; ct >>= 1)
    if (batch_tiles > 1 && cols % ct == 0 && cols / ct * batch_tiles >= kWorkgroups) return ct;
  return 1;
}

// Mixed mode: whether a projection of `cols` column tiles folds its norm. Folded, it saves the norm's
// kernel and converts its X rows again in each group of column tiles; behind the norm's kernel it
// takes X in FP16, four batch tiles to a workgroup. So it folds where there are no four tiles, else up
// to a line of values converted, rows x K x groups. us per layer of the fold against the norm's kernel,
// swept over widths 256 to 1024, ffn 256 to 4096 and 1 to 256 streams: up to 32 streams always
// less (-1.1 to -2.6). From 64 on, gate/up at 4.2 M -3.9 to -1.3, 8.4 M -1.0 to -0.1, 12.6 M -0.3 to
// +1.1, 16.8 M +2.8 and +3.4; QKV at 6.3 M -1.4 and -1.2, 9.4 M -0.1 to +0.4, 12.6 M -0.1 and +0.3. Odd
// column tile counts, whose four-tile shape shares X with no second column tile: 11.3 M -0.8, 12.3 M
// +0.6, 14.2 M +0.3, 16.7 M +2.1. Odd numbers of groups of four tiles lose sooner at the wider K:
// 3.5 M and 3.9 M -1.6, 4.3 M to 5.9 M at 128 rows +0.7 to +2.0, 6.5 M +0.4 to +0.9 (at K = 512 still
// -1.2 at 4.3 M, -1.1 at 4.9 M).
bool Batch::folds_norm(int cols) const {
  const int ct = column_tiles(cols), groups = cols / ct;
  const size_t line = (size_t)(cols % 2 ? 12 : ct == 4 && groups % 2 && args_.width_p > 512 ? 4 : 8) << 20;
  return streams_p_ % (4 * kBatchTile) != 0 || (size_t)streams_p_ * args_.width_p * groups <= line;
}

// One projection. Every workgroup shape computes the same fixed slice tree, so the choice changes
// speed only, never a stream's bits. Each workgroup re-reads its rows of X and its rows of the
// weights, and converts X to MFMA operands, so more column tiles (CT) share both; the chip wants
// about as many workgroups as it has CUs. So CT is the largest of 4, 2, 1 that leaves kWorkgroups,
// with one batch tile (NT): us per layer against two K-slices per wave and 1 to 4 batch tiles, the
// shapes of before, gate/up 4 x 1 -3.1 for Large at 32 streams, -12.2 at 128, -0.8 for Main at 64;
// QKV 2 x 1 -1.2 for Large at 32, 4 x 1 -4.4 at 128; narrow projections of small models (128 tiles)
// 1 x 1 instead of 2 x 1 -1.3 for Small at 100. At one batch tile a wider CT gains nothing (Large
// at 8 streams, gate/up 2 x 1 +0.1 to +0.5).
// Mixed mode's norm kernels hand over X in FP16: nothing to convert, and weights are most of the
// traffic, so four batch tiles share them (2 x 4: Large at 128 streams, QKV -1.1 and gate/up -3.4
// against 4 x 1; at 256 -1.0 and -2.4; odd column tile counts 1 x 4: 173 of gate/up at 192 streams
// -3.4 against 1 x 1, 105 of QKV at 128 -2.1).
template <int P, int E, bool kNorm>
void Batch::project(const void* X, int ld, void* out, int out_ld, uint32_t woff, int N, uint32_t norm, int layer) {
  const int cols = N / kBatchTile, batch_tiles = streams_p_ / kBatchTile;
  // Blocks in flight per wave (k_ring): four where a slice holds a multiple of four, else two.
  constexpr int kb = P == kFp32 || (P == kMixed && E == kEpInput) ? 16 : 32;
  const bool deep = ld / kSlices / kb % 4 == 0;
  auto go = [&](auto kernel, int nt, int ct) {
    hipLaunchKernelGGL(kernel, dim3(cols / ct, batch_tiles / nt), dim3(64 * kSlices), 0, stream_, args_.weights, X, out,
                       dargs_, woff, ld, norm, c_.width, streams_, out_ld, layer);
  };
  if constexpr (P == kMixed && !kNorm && (E == kEpQkv || E == kEpGateUp)) {
    if (cols % 2 == 0) go(batch_proj<P, E, kNorm, 4, 2, 2>, 4, 2);
    else go(batch_proj<P, E, kNorm, 4, 1, 2>, 4, 1);
  } else {
    const int ct = E == kEpInput ? 1 : column_tiles(cols);
    if constexpr (E != kEpInput) {
      if (ct == 4) return go(batch_proj<P, E, kNorm, 1, 4, 2>, 1, 4);
      if (ct == 2) return deep ? go(batch_proj<P, E, kNorm, 1, 2, 4>, 1, 2) : go(batch_proj<P, E, kNorm, 1, 2, 2>, 1, 2);
    }
    if (deep) go(batch_proj<P, E, kNorm, 1, 1, 4>, 1, 1);
    else go(batch_proj<P, E, kNorm, 1, 1, 2>, 1, 1);
  }
}

// Attention of one layer. Windows of more than one chunk: a workgroup per (stream, head, chunk)
// where the (stream, head) pairs alone give fewer than kSplitPairs workgroups, else one that walks
// its chunks. Below the line the spread fills the chip: us per step of two layers, split / walked,
// at 32 pairs 52.8 / 60.7 (FP16 K/V, eight chunks) and 80.2 / 97.7 (FP32, 16 chunks, head dim 128),
// at 128 pairs 60.5 / 62.7 and 142.9 / 144.2. From the line on the partials written, counted and
// read back cost more than that gives: at 192 pairs 64.0 / 64.5 and 187.6 / 169.7, with 32 chunks
// 216.0 / 170.3 (FP32, head dim 64), at 512 pairs of 16 chunks 236 / 205. A few pairs more than one
// per CU put two walks on a few CUs, which the others wait for: at 264 pairs 68.8 / 75.5 (FP16, eight
// chunks), 95.8 / 104.1 and 150.3 / 160.8 (FP32, eight and 16); even at 320, 72.8 / 76.4, 106.3 / 107.7 and
// 169.7 / 166.5. Two chunks are walked there too (62.6 / 62.0, head dim 128 75.3 / 73.9; three 67.0 / 68.1
// and 87.9 / 89.7).
template <int P, bool kNT>
void Batch::attend(int layer) {
  const size_t block = (size_t)c_.width * c_.window * (P == kMixed ? 2 : 4);  // a (layer, stream) block in bytes
  const char* keys = reinterpret_cast<const char*>(args_.keys) + (size_t)layer * streams_ * block;
  const char* values = reinterpret_cast<const char*>(args_.values) + (size_t)layer * streams_ * block;
  if (dim_ > 128) {
    hipLaunchKernelGGL((batch_attention_wide<P, kNT>), dim3(c_.heads, streams_), dim3(kAttnThreads), (size_t)c_.window * 4,
                       stream_, args_.position, args_.q, keys, values, args_.attn, c_.window, dim_, c_.heads, args_.width_p);
    return;
  }
  const int chunks = attn_chunks();
  const bool split = attn_split();
  auto go = [&](auto kernel, int dv) {
    const size_t lds = (size_t)(split ? 1 : chunks) * kAttnWaves * (64 * dv + 2) * 4;
    hipLaunchKernelGGL(kernel, dim3(c_.heads, streams_, split ? chunks : 1), dim3(kAttnThreads), lds, stream_, args_.position,
                       args_.q, keys, values, args_.attn, c_.window, dim_, c_.heads, args_.width_p,
                       reinterpret_cast<float*>(attn_part_.ptr), reinterpret_cast<unsigned*>(attn_count_.ptr));
  };
  // The loads that do not wait for the position read every slot of the window: for one-chunk
  // windows whose rings stay cached and that are too few to fill the chip (elsewhere the unwritten
  // slots' bytes would cost more than the round trip).
  const bool any = !kNT && chunks == 1 && streams_ * c_.heads <= kCuPairs;
  auto form = [&](auto DV, auto NP) {
    constexpr int dv = decltype(DV)::value, np = decltype(NP)::value;
    if constexpr (!kNT) {
      if (any) return go(batch_attention<P, dv, np, true, kNT>, dv);
    }
    go(batch_attention<P, dv, np, false, kNT>, dv);
  };
  using std::integral_constant;
  if (dim_ > 64) {
    if (c_.window <= 64) form(integral_constant<int, 2>{}, integral_constant<int, 4>{});
    else form(integral_constant<int, 2>{}, integral_constant<int, 8>{});
  } else {
    if (c_.window <= 64) form(integral_constant<int, 1>{}, integral_constant<int, 4>{});
    else form(integral_constant<int, 1>{}, integral_constant<int, 8>{});
  }
}

template <int P>
void Batch::launch_sequence() {
  const BatchArgs& a = args_;
  const int d = c_.width, F = c_.ffn;
  // K/V rings that do not fit in the Infinity Cache beside the weights are read with
  // non-temporal loads, so that the weights stay cached.
  const bool kv_nt = 2 * c_.layers * (size_t)streams_ * block_words_ * 4 + offsets_.weight_bytes > kInfinityCacheBytes;
  // The norms are folded into the projections (kNorm), or run first, into xn. Main's mixed steps
  // without the fold and with it: 167.7 -> 142.9 us at one stream, 177 -> 144 at 16, 200 -> 177 at 64.
  const bool fold_qkv = P != kMixed || folds_norm(3 * d / kBatchTile);
  const bool fold_gateup = P != kMixed || folds_norm(2 * F / kBatchTile);
  auto qkv = [&](const LayerWeights& w, int l, const void* x, auto kFold) {
    project<P, kEpQkv, decltype(kFold)::value>(x, a.width_p, nullptr, 0, w.qkv, 3 * d, w.norm1, l);
  };
  auto gateup = [&](const LayerWeights& w, int l, const void* x, auto kFold) {
    project<P, kEpGateUp, decltype(kFold)::value>(x, a.width_p, a.act, a.ffn_p, w.gateup, 2 * F, w.norm2, l);
  };
  auto normed = [&](auto&& projection, const LayerWeights& w, uint32_t w_norm, int l, bool fold) {
    if constexpr (P == kMixed) {
      if (!fold) {
        hipLaunchKernelGGL(batch_norm_mixed, dim3(streams_p_), dim3(256), 0, stream_, dargs_, w_norm);
        return projection(w, l, a.xn, std::false_type{});
      }
    }
    projection(w, l, a.x, std::true_type{});
  };
  project<P, kEpInput, false>(a.in, a.features_p, a.x, a.width_p, a.w_input, d, 0u, 0);
  for (int l = 0; l < c_.layers; l++) {
    const LayerWeights& w = a.layer[l];
    normed(qkv, w, w.norm1, l, fold_qkv);
    if (kv_nt) attend<P, true>(l);
    else attend<P, false>(l);
    project<P, kEpOut, false>(a.attn, a.width_p, a.x, a.width_p, w.out, d, 0u, l);
    normed(gateup, w, w.norm2, l, fold_gateup);
    project<P, kEpDown, false>(a.act, a.ffn_p, a.x, a.width_p, w.down, d, 0u, l);
  }
  hipLaunchKernelGGL(batch_final<P>, dim3(streams_), dim3(64), 0, stream_, dargs_);
  HIP_CHECK(hipGetLastError());
}

// The events of one step into the padded input block in the projections' operand layout.
// Four consecutive columns from a multiple of 4 are consecutive in the layout.
void Batch::stage_events(const float* inputs, float* block) const {
  const int fp = args_.features_p;
  auto at = [&](int b, int k) { return prec_ == kBf16w ? act_index<kBf16w>(b, k, fp) : act_index<kFp32>(b, k, fp); };
  for (int b = 0; b < streams_; b++) {
    const float* src = inputs + (size_t)b * c_.features;
    int k = 0;
    for (; k + 4 <= c_.features; k += 4) std::memcpy(block + at(b, k), src + k, 16);
    for (; k < c_.features; k++) block[at(b, k)] = src[k];
  }
}

// The events go to mapped host memory as they come; batch_stage reads them there and lays them out,
// and the last kernel writes the scores to mapped host memory: no copy command on either side.
// Pieces of kStageBytes, so that the host copies one while the device reads the one before. With
// copy commands and the layout done here by the host, a step took longer than its kernels by
// 25 us for Main at 16 streams, 35 at 64 and 63 at 256; now by 14, 20 and 41.
void Batch::step(const float* inputs, float* scores) {
  if (!inputs || !scores) throw Error(ST_ERR_INVALID, "Null argument");
  constexpr size_t kStageBytes = 128 << 10;
  const int F = c_.features;
  float* h = reinterpret_cast<float*>(host_in_.ptr);
  const int most = (int)std::max<size_t>(1, kStageBytes / ((size_t)F * 4));
  for (int b = 0; b < streams_; b += most) {
    const int rows = std::min(most, streams_ - b);
    std::memcpy(h + (size_t)b * F, inputs + (size_t)b * F, (size_t)rows * F * 4);
    const dim3 grid((rows * ((F + 3) / 4) + 255) / 256);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream_, reinterpret_cast<const float*>(host_in_.dev), args_.in, b, rows,
                         F, args_.features_p);
    };
    if (prec_ == kBf16w) go(batch_stage<kBf16w>);
    else go(batch_stage<kFp32>);
    HIP_CHECK(hipGetLastError());
  }
  replay();
  sync();
  std::memcpy(scores, host_out_.ptr, (size_t)streams_ * 4);
}

void Batch::reset(int stream) {
  if (stream < -1 || stream >= streams_) throw Error(ST_ERR_INVALID, "Stream index out of range");
  hipLaunchKernelGGL(batch_reset, dim3(256), dim3(256), 0, stream_, dargs_, stream, block_words_);
  HIP_CHECK(hipGetLastError());
  sync();
}

void Batch::snapshot(int stream, uint64_t* position, float* keys, float* values, float* hidden) {
  if (stream < 0 || stream >= streams_) throw Error(ST_ERR_INVALID, "Stream index out of range");
  sync();
  const size_t ring = (size_t)c_.layers * c_.width * c_.window;
  if (position)
    HIP_CHECK(hipMemcpy(position, args_.position + stream, 8, hipMemcpyDeviceToHost));
  // The stream's block of each layer (layer-major rings) into [L][H][W][dh].
  auto download = [&](const void* base, float* dst) {
    if (!dst) return;
    const size_t block = block_words_ * 4, pitch = (size_t)streams_ * block;
    const char* src = reinterpret_cast<const char*>(base) + (size_t)stream * block;
    if (prec_ == kMixed) {
      std::vector<uint16_t> h(ring);
      HIP_CHECK(hipMemcpy2D(h.data(), block, src, pitch, block, c_.layers, hipMemcpyDeviceToHost));
      for (size_t i = 0; i < ring; i++) dst[i] = host_half_to_float(h[i]);
    } else {
      HIP_CHECK(hipMemcpy2D(dst, block, src, pitch, block, c_.layers, hipMemcpyDeviceToHost));
    }
  };
  download(args_.keys, keys);
  download(args_.values, values);
  if (hidden)
    HIP_CHECK(hipMemcpy(hidden, args_.hidden + (size_t)stream * c_.layers * c_.width, (size_t)c_.layers * c_.width * 4,
                        hipMemcpyDeviceToHost));
}

// `count` batched steps from a preloaded device copy of the inputs (count x streams x
// features), continuing the current state; one graph replay per step after a device-to-device
// copy of that step's inputs, with a HIP event after each. Returns the mean microseconds per
// step and, when per_step is not NULL, each step's event-to-event duration.
double Batch::device_run(const float* inputs, size_t count, double* per_step) {
  const int fp = args_.features_p;
  // The padded copy is staged on the host and the device: at most 4 GiB.
  if (!inputs || count == 0 || count > ((size_t)1 << 30) / ((size_t)streams_p_ * fp))
    throw Error(ST_ERR_INVALID, "Invalid trace (empty, or more than 4 GiB of padded inputs)");
  std::vector<float> padded(count * (size_t)streams_p_ * fp, 0.f);
  for (size_t i = 0; i < count; i++)
    stage_events(inputs + i * streams_ * c_.features, &padded[i * streams_p_ * fp]);
  DeviceBuffer dev;
  dev.alloc(padded.size() * 4);
  HIP_CHECK(hipMemcpy(dev.ptr, padded.data(), padded.size() * 4, hipMemcpyHostToDevice));
  std::vector<hipEvent_t> ev(count + 1);
  for (auto& e : ev) create_timing_event(&e);
  sync();
  HIP_CHECK(hipEventRecord(ev[0], stream_));
  for (size_t i = 0; i < count; i++) {
    HIP_CHECK(hipMemcpyAsync(args_.in, reinterpret_cast<float*>(dev.ptr) + i * (size_t)streams_p_ * fp,
                             (size_t)streams_p_ * fp * 4, hipMemcpyDeviceToDevice, stream_));
    replay();
    HIP_CHECK(hipEventRecord(ev[i + 1], stream_));
  }
  sync();
  double total = 0;
  for (size_t i = 0; i < count; i++) {
    float ms = 0;
    HIP_CHECK(hipEventElapsedTime(&ms, ev[i], ev[i + 1]));
    if (per_step) per_step[i] = ms * 1000.0;
    total += ms * 1000.0;
  }
  for (auto& e : ev) (void)hipEventDestroy(e);
  return total / count;
}

}  // namespace stamd
