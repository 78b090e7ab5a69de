#include "blaze/predictor.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <type_traits>

#include "blaze/feed_pack.h"
#include "blaze/qed_store.h"
#include "blaze_hip.h"

namespace blaze {

Predictor::Predictor(std::shared_ptr<Net> net) : net_(net) {
  for (const auto& name : net_->external_output()) {
    Blob* b = net_->external_output_blob(name);
    BLAZE_CONDITION_THROW(b != nullptr, "external_output: ", name, " is not in external_output_blob");
    output_index_[name] = (int)external_output_blob_.size();
    external_output_blob_.push_back(b);
    DeviceOption cpu;
    cpu.set_device_type(kCPU);
    output_cpu_.push_back(std::make_shared<Blob>(cpu));
    output_cpu_.back()->set_data_type((DataType)b->data_type());
  }
  output_wanted_.assign(output_cpu_.size(), false);
  output_ahead_.assign(output_cpu_.size(), false);
  output_by_operator_.assign(output_cpu_.size(), false);
  output_half_.assign(output_cpu_.size(), 0);
  output_read_.assign(output_cpu_.size(), 0);
  output_pinned_.assign(output_cpu_.size(), false);
  for (Blob* b : external_output_blob_) {
    int writers = 0, readers = 0;
    for (const auto& op : net_->GetOperators()) {
      // (a constant's blob is every predictor's: nothing of one pass is kept in it)
      for (int i = 0; i < op->OutputSize(); ++i) writers += op->Output(i) == b && op->type() != "ConstantFill";
      for (int i = 0; i < op->InputSize(); ++i) readers += op->Input(i) == b;
    }
    output_sole_.push_back(writers == 1 && readers == 0);
  }
  await_outputs_ = EveryOperatorFeedsAnOutput();
  for (const auto& name : net_->external_input()) {
    Blob* b = net_->external_input_blob(name);
    BLAZE_CONDITION_THROW(b != nullptr, "external_input: ", name, " is not in external_input_blob");
    input_index_[name] = (int)external_input_blob_.size();
    external_input_blob_.push_back(b);
    DeviceOption cpu;
    cpu.set_device_type(kCPU);
    input_cpu_.push_back(std::make_shared<Blob>(cpu));
    feed_pending_.push_back(false);
  }
}

Predictor::~Predictor() {
  // Wait only for work that is still queued: an event that was already waited for may belong to a stream that died with
  // its serving thread.  Nothing here may leave an error behind for the caller's next runtime call.
  if (any_feed_pending_ && feed_recorded_) (void)hipEventSynchronize(feed_done_);
  if ((any_feed_pending_ && !feed_recorded_) || !settled_) (void)WaitForDevice();
  if (forward_done_ && forward_in_flight_) (void)hipEventSynchronize(forward_done_);
  if (arena_host_) (void)hipHostFree(arena_host_);
  if (arena_dev_) (void)hipFree(arena_dev_);
  for (void* a : retired_arenas_) (void)hipFree(a);
  if (forward_done_) (void)hipEventDestroy(forward_done_);
  if (feed_done_) (void)hipEventDestroy(feed_done_);
  (void)hipGetLastError();
}

// All streams of this predictor's device have been waited for, whatever device the calling thread is on.
hipError_t Predictor::WaitForDevice() const {
  int before = 0;
  hipError_t rc = hipGetDevice(&before);
  const int mine = device_id();
  if (rc == hipSuccess && mine >= 0) rc = hipSetDevice(mine);
  if (rc == hipSuccess) rc = hipDeviceSynchronize();
  if (mine >= 0 && mine != before) (void)hipSetDevice(before);
  return rc;
}

int Predictor::InputName2Idx(const char* name) const {
  auto it = input_index_.find(name);
  return it == input_index_.end() ? -1 : it->second;
}
int Predictor::OutputName2Idx(const char* name) const {
  auto it = output_index_.find(name);
  return it == output_index_.end() ? -1 : it->second;
}

bool Predictor::ReshapeInput(const char* name, const std::vector<size_t>& shape) {
  const int idx = InputName2Idx(name);
  if (idx < 0) {
    LOG_ERROR("The name: %s is not The input of net", name);
    return false;
  }
  return ReshapeInput((size_t)idx, shape);
}
bool Predictor::ReshapeInput(size_t idx, const std::vector<size_t>& shape) {
  if (idx >= external_input_blob_.size()) {
    LOG_ERROR("The idx=%zu exceed size=%zu", idx, external_input_blob_.size());
    return false;
  }
  output_ahead_.assign(output_ahead_.size(), false);  // (an input may itself be an output, of another size from here on)
  try {
    external_input_blob_[idx]->Reshape(shape);
  } catch (std::exception& e) {
    LOG_ERROR("reshape failed: %s", e.what());
    return false;
  }
  return true;
}

namespace {
// rows of a 2-D input that lives inside a Concat's output, from a dense staging copy
bz_feed_rows StridedRows(Blob* blob, const void* staged) {
  const int64_t es = (int64_t)DataTypeSize(blob->data_type()), w = (int64_t)blob->shape()[1] * es;
  bz_feed_rows r;
  r.src = staged;
  r.dst = blob->data();
  r.rows = (int64_t)blob->shape()[0];
  r.row_bytes = r.src_pitch = w;
  r.dst_pitch = (int64_t)blob->pitch() * es;
  return r;
}
}  // namespace

bool Predictor::Feed(const char* name, const void* data, size_t len) {
  const int idx = InputName2Idx(name);
  if (idx < 0) {
    LOG_ERROR("The name: %s is not The input of net", name);
    return false;
  }
  return Feed((size_t)idx, data, len);
}
bool Predictor::Feed(size_t idx, const void* data, size_t len) {
  if (idx >= external_input_blob_.size()) {
    LOG_ERROR("The idx=%zu exceed size=%zu", idx, external_input_blob_.size());
    return false;
  }
  output_ahead_.assign(output_ahead_.size(), false);  // (an input may itself be an output)
  Blob* blob = external_input_blob_[idx];
  const size_t need = blob->size() * DataTypeSize(blob->data_type());
  if (len != need) {
    LOG_ERROR("The len=%zu need size=%zu blob->size()=%zu", len, need, (size_t)blob->size());
    return false;
  }
  try {
    if (blob->device_type() == kCPU) {
      memcpy(blob->data(), data, need);
    } else {
      HIPContext ctx(blob->device_option());
      ctx.Activate();
      hipStream_t st = ctx.hip_stream();
      if (blob->unplaced()) {  // outgrew its slice of the FeedMany arena: back to memory of its own
        const std::vector<TIndex> shape = blob->shape();
        blob->DropArenaView();
        blob->Reshape(shape);
      }
      SettleBefore(ctx);
      // stage in pinned memory and queue the transfer; a second Feed of the same input first waits for the first
      if (feed_done_ == nullptr) HIP_CHECK(hipEventCreateWithFlags(&feed_done_, hipEventDisableTiming));
      if (feed_pending_[idx]) FinishFeeds();
      Blob* stage = input_cpu_[idx].get();
      stage->set_data_type((DataType)blob->data_type());
      stage->Reshape(blob->shape());
      memcpy(stage->data(), data, need);
      if (blob->pitch() != 0) {  // the input lives inside a Concat's output: rows are `pitch` elements apart
        const bz_feed_rows r = StridedRows(blob, stage->data());
        if (IsPinnedHost(stage->data()))
          BZ_CHECK(bz_feed(nullptr, nullptr, 0, &r, 1, st));
        else  // (staging the runtime could not pin: a kernel cannot read it)
          HIP_CHECK(hipMemcpy2DAsync(r.dst, r.dst_pitch, r.src, r.src_pitch, r.row_bytes, r.rows, hipMemcpyHostToDevice, st));
      } else if (need > 0) {
        HIP_CHECK(hipMemcpyAsync(blob->data(), stage->data(), need, hipMemcpyHostToDevice, st));
      }
      FeedQueued(ctx);
      feed_pending_[idx] = true;
    }
  } catch (std::exception& e) {
    LOG_ERROR("feed failed: %s", e.what());
    return false;
  }
  return true;
}

// a transfer has been queued on the context's stream
void Predictor::FeedQueued(const HIPContext& ctx) {
  feed_on_ = ctx.stream_serial();
  feed_recorded_ = feed_on_ != forward_on_;
  if (feed_recorded_) HIP_CHECK(hipEventRecord(feed_done_, ctx.hip_stream()));
  any_feed_pending_ = true;
}

// The queued transfers have ended.  Without an event, from another thread: the stream they are on may be gone with its thread,
// the device is not.
void Predictor::FinishFeeds() {
  if (feed_recorded_) {
    HIP_CHECK(hipEventSynchronize(feed_done_));
  } else {
    for (Blob* b : external_input_blob_) {
      if (b->device_type() != kHIP) continue;
      HIPContext ctx(b->device_option());
      ctx.Activate();
      HIP_CHECK(ctx.stream_serial() == feed_on_ ? hipStreamSynchronize(ctx.hip_stream()) : WaitForDevice());
      break;
    }
  }
  std::fill(feed_pending_.begin(), feed_pending_.end(), false);
  any_feed_pending_ = false;
}

// what this thread launches from here on runs behind the queued transfers, and behind the last pass
void Predictor::OrderBehindFeeds() {
  for (const auto* list : {&external_input_blob_, &external_output_blob_})
    for (Blob* b : *list) {
      if (b->device_type() != kHIP) continue;
      HIPContext ctx(b->device_option());
      ctx.Activate();
      SettleBefore(ctx);
      forward_on_ = ctx.stream_serial();
      if (!any_feed_pending_ || forward_on_ == feed_on_) return;
      if (feed_recorded_)
        HIP_CHECK(hipStreamWaitEvent(ctx.hip_stream(), feed_done_, 0));
      else
        HIP_CHECK(WaitForDevice());
      return;
    }
}

bool Predictor::FeedMany(int count, const char* const* names, const void* const* data, const size_t* lens) {
  output_ahead_.assign(output_ahead_.size(), false);
  try {
    struct Item : FeedInput {
      int idx;
    };
    struct Strided {
      int idx;
      int arg;
      size_t offset;
    };
    // plain inputs first, in one range that lands as it is staged; inputs that live inside a Concat's output behind them
    std::vector<Item> in_arena;
    in_arena.reserve(std::max(count, 0));
    std::vector<Strided> strided;
    size_t total = 0;
    const DeviceOption* dev = nullptr;
    for (int i = 0; i < count; ++i) {
      const int idx = InputName2Idx(names[i]);
      if (idx < 0) {
        LOG_ERROR("The name: %s is not The input of net", names[i]);
        return false;
      }
      Blob* blob = external_input_blob_[idx];
      const size_t word = DataTypeSize(blob->data_type()), need = blob->size() * word;
      if (lens[i] != need) {
        LOG_ERROR("The len=%zu need size=%zu blob->size()=%zu", lens[i], need, (size_t)blob->size());
        return false;
      }
      if (blob->device_type() != kHIP) {
        if (!Feed((size_t)idx, data[i], lens[i])) return false;
        continue;
      }
      dev = &blob->device_option();
      if (blob->pitch() != 0) {
        auto same = std::find_if(strided.begin(), strided.end(), [&](const Strided& it) { return it.idx == idx; });
        if (same != strided.end())
          same->arg = i;  // named twice: the last one counts, and two pieces of one launch must not share a target
        else
          strided.push_back({idx, i, 0});
        continue;
      }
      in_arena.push_back({{data[i], need, total, word}, idx});
      total += (need + 255) / 256 * 256;  // every slice 256-byte aligned
    }
    if (dev == nullptr) return true;
    const size_t plain = total;
    for (Strided& it : strided) {
      it.offset = total;
      total += (lens[it.arg] + 255) / 256 * 256;
    }
    HIPContext ctx(*dev);
    ctx.Activate();
    SettleBefore(ctx);
    hipStream_t st = ctx.hip_stream();
    if (feed_done_ == nullptr) HIP_CHECK(hipEventCreateWithFlags(&feed_done_, hipEventDisableTiming));
    if (any_feed_pending_) FinishFeeds();  // the staging arena may still be read by the previous transfer
    if (total > arena_cap_) {
      if (arena_host_) HIP_CHECK(hipHostFree(arena_host_));
      if (arena_dev_) retired_arenas_.push_back(arena_dev_);
      arena_host_ = arena_dev_ = nullptr;
      arena_cap_ = 0;
      const size_t cap = total + total / 4;
      AllocationCount() += 2;
      HIP_CHECK(hipHostMalloc((void**)&arena_host_, cap, hipHostMallocDefault));
      HIP_CHECK(hipMalloc((void**)&arena_dev_, cap));
      arena_cap_ = cap;
    }
    // from the first launch on the arena is being read: whatever happens next, it is waited for before it is written again
    try {
      bz_feed_rows rows[BZ_FEED_MAX_ROWS];
      int n = 0;
      auto launch = [&](const bz_feed_piece* pieces, int n_pieces) {
        BZ_CHECK(bz_feed_pieces(pieces, n_pieces, rows, n, st));
        n = 0;
      };
      for (const Strided& it : strided) {
        if (n == BZ_FEED_MAX_ROWS) launch(nullptr, 0);
        memcpy(arena_host_ + it.offset, data[it.arg], lens[it.arg]);
        rows[n++] = StridedRows(external_input_blob_[it.idx], arena_host_ + it.offset);
      }
      StageInputs(in_arena, plain, arena_host_, arena_dev_, launch);
      if (n > 0) launch(nullptr, 0);
      FeedQueued(ctx);
    } catch (...) {
      (void)hipStreamSynchronize(st);  // no event stands behind what was launched
      any_feed_pending_ = false;
      throw;
    }
    for (const Strided& it : strided) feed_pending_[it.idx] = true;
    for (const Item& it : in_arena) {
      Blob* blob = external_input_blob_[it.idx];
      // (also when the slice did not move: this records the slice's new size and clears "unplaced")
      const std::vector<TIndex> shape = blob->shape();
      blob->RefReshape(shape, arena_dev_ + it.offset, /*arena_view=*/true);
      feed_pending_[it.idx] = true;
    }
  } catch (std::exception& e) {
    LOG_ERROR("feed failed: %s", e.what());
    last_error_for_thread() = e.what();
    return false;
  }
  return true;
}

int Predictor::InputDataType(const char* name) const {
  const int idx = InputName2Idx(name);
  return idx < 0 ? (int)kPDT_Invalid : external_input_blob_[idx]->data_type();
}

int Predictor::device_id() const {
  for (const auto* list : {&external_output_blob_, &external_input_blob_})
    for (Blob* b : *list)
      if (b->device_type() == kHIP) return b->device_option().device_id();
  return -1;
}

bool Predictor::ForwardLaunch() {
  try {
    for (size_t i = 0; i < external_input_blob_.size(); ++i)
      if (external_input_blob_[i]->unplaced()) {
        last_error_for_thread() = "input " + net_->external_input()[i] + " was reshaped beyond its fed size and has not been fed since";
        LOG_ERROR("%s", last_error_for_thread().c_str());
        return false;
      }
    OrderBehindFeeds();
    output_ahead_.assign(output_ahead_.size(), false);
    if (!net_->Launch()) return false;
    launched_on_ = net_->StreamOfLastLaunch();
    if (launched_on_ != nullptr) {
      if (forward_done_ == nullptr) HIP_CHECK(hipEventCreateWithFlags(&forward_done_, hipEventDisableTiming));
      HIP_CHECK(hipEventRecord(forward_done_, (hipStream_t)launched_on_));
    }
    forward_in_flight_ = true;
    return true;
  } catch (std::exception& e) {
    LOG_ERROR("failed: %s", e.what());
    last_error_for_thread() = e.what();
    return false;
  }
}

bool Predictor::ForwardWait() {
  try {
    if (!forward_in_flight_) {
      last_error_for_thread() = "ForwardWait without a ForwardLaunch before it";
      return false;
    }
    forward_in_flight_ = false;
    // the event sits behind the net's last operator, which sits behind the queued input transfers
    if (launched_on_ != nullptr) HIP_CHECK(hipEventSynchronize(forward_done_));
    if (any_feed_pending_) {
      std::fill(feed_pending_.begin(), feed_pending_.end(), false);
      any_feed_pending_ = false;
    }
    return true;
  } catch (std::exception& e) {
    LOG_ERROR("failed: %s", e.what());
    last_error_for_thread() = e.what();
    return false;
  }
}

bool Predictor::Forward(const PredictorCallback&& cb) {
  try {
    if (forward_in_flight_ && !ForwardWait()) return false;  // a launch the caller never waited for
    for (size_t i = 0; i < external_input_blob_.size(); ++i)
      if (external_input_blob_[i]->unplaced()) {
        last_error_for_thread() = "input " + net_->external_input()[i] + " was reshaped beyond its fed size and has not been fed since";
        LOG_ERROR("%s", last_error_for_thread().c_str());
        return false;
      }
    OrderBehindFeeds();
    output_ahead_.assign(output_ahead_.size(), false);
    output_by_operator_.assign(output_by_operator_.size(), false);
    awaited_.clear();
    OfferHostCopies();
    const bool launched = net_->Launch();
    if (launched) QueueOutputs();
    WithdrawHostCopies();
    if (!launched) return false;
    settled_ = false;
    if (!PassIsThere()) {
      net_->Wait();
      settled_ = true;
      passes_unsettled_ = 0;
    }
    if (any_feed_pending_) {  // Run waited for the stream, which had waited for the transfers
      std::fill(feed_pending_.begin(), feed_pending_.end(), false);
      any_feed_pending_ = false;
    }
    if (cb) cb();
    return true;
  } catch (std::exception& e) {
    WithdrawHostCopies();
    output_ahead_.assign(output_ahead_.size(), false);
    LOG_ERROR("failed: %s", e.what());
    last_error_for_thread() = e.what();
    return false;
  }
}

namespace {
// whether two blobs share memory (an output may be an input, or a Reshape's view of one)
bool Overlap(Blob* a, Blob* b) {
  auto range = [](Blob* x, uintptr_t* from, uintptr_t* to) {
    const size_t es = DataTypeSize(x->data_type());
    *from = (uintptr_t)x->data();
    *to = *from + x->size() * es;
    if (x->pitch() != 0 && x->size() > 0) *to = *from + ((x->shape()[0] - 1) * x->pitch() + x->shape()[1]) * es;
  };
  uintptr_t a0, a1, b0, b1;
  range(a, &a0, &a1);
  range(b, &b0, &b1);
  return a0 < b1 && b0 < a1;
}
}  // namespace

// Outputs that were read after the last Forward are copied to the host behind this one, under the same wait: a copy asked
// for by Output alone is another launch and another wait, 16 us of a 58 us request.  Small ones only, by a kernel that
// writes the pinned copy over the link (the copy engine's hand-over would cost more than it moves); larger ones are
// copied by Output.  Into the other half of the host buffer: the half Output handed out stays as it is until the next Output.
// Not where the caller holds the device address of that memory: what it writes there after the pass is the output, too.
// Output makes both halves in one allocation (one between a launch and its wait would hold the pass up), so an output that
// has grown since is copied by Output once more.
constexpr size_t kCopiedAheadMax = 64 << 10;
constexpr TIndex kHalfAlign = 64;  // elements

size_t Predictor::HostHalf(size_t i) const {
  const Blob& b = *output_cpu_[i];
  return b.capacity() / (2 * kHalfAlign) * kHalfAlign * DataTypeSize(b.data_type());
}

// whether output i may be copied ahead as far as one can say without its size
bool Predictor::CopiedAhead(size_t i) const {
  Blob* blob = external_output_blob_[i];
  if (!output_wanted_[i] || blob->device_type() != kHIP || output_cpu_[i]->data_type() != blob->data_type() || HostHalf(i) < output_read_[i] ||
      !output_pinned_[i])
    return false;
  return std::none_of(handed_out_.begin(), handed_out_.end(), [&](Blob* b) { return Overlap(b, blob); });
}

// A small output that comes as floats is known to have arrived when no element has the value any more that was there before the
// launch: all bits set, a NaN that no operator makes of its own.
constexpr int kNotThereByte = 0xff;

// Before the launches: the operator that writes such an output may write the copy in the same launch (a layer's skinny head,
// bz::fc_fused).  A launch behind it is 2 to 4 us of a request: one sample fp32 40.3 -> 38.3, 300 samples fp16 60.8 -> 57.1,
// the attention model at 1024 105..114 -> 102.  Only where nothing else in the net touches the output.
void Predictor::OfferHostCopies() {
  for (size_t i = 0; i < external_output_blob_.size(); ++i) {
    if (!output_sole_[i] || !CopiedAhead(i)) continue;
    Blob::HostCopy& c = external_output_blob_[i]->host_copy();
    c.copied = 0;
    c.room = std::min(HostHalf(i), kCopiedAheadMax);
    c.at = (char*)output_cpu_[i]->data() + (1 - output_half_[i]) * HostHalf(i);
    c.fill = Awaitable(i) ? kNotThereByte : -1;
  }
}

bool Predictor::Awaitable(size_t i) const {
  const int dt = output_cpu_[i]->data_type();
  return await_outputs_ && (dt == kFloat || dt == kFloat16);
}

// Whether the pass has ended, as far as anybody but a stream can tell: every output is on its way to the host by itself, and
// all of it has arrived.  The stream behind it need not be waited for, which is a packet on the queue and the runtime's own
// turn: 4.6 us of a chain of four small launches of 19.1.  What runs on the device still is the end of the launches whose results
// have arrived, since every operator's reach an output (EveryOperatorFeedsAnOutput).  What this thread queues is behind that on the
// stream; who goes round the stream waits first: a feed or a pass on another one (SettleBefore), a device address, a copy by Output,
// the destructor (Settle); and memory that is freed waits for the device by itself.  Every 32nd pass waits for the stream, so
// that the runtime can put away what it keeps for each launch (left alone it does so every thousand or so, in 5 ms).
// us a request, with the event that is no longer recorded behind the transfer: one sample fp32 35.5 -> 32.0, 300 samples fp16
// 50.7 -> 45.2, attention models of 201 and 1024 59.2 -> 52.7 and 101.6 -> 93.7, 2048 samples 230 -> 209.
constexpr int kSettleEvery = 32;
constexpr auto kAwaitAtMost = std::chrono::microseconds(300);
bool Predictor::PassIsThere() {
  if (awaited_.size() != external_output_blob_.size() || awaited_.empty() || ++passes_unsettled_ >= kSettleEvery) return false;
  const auto t0 = std::chrono::steady_clock::now();
  auto arrived = [&](auto* p, size_t n) {
    typedef std::remove_cv_t<std::remove_pointer_t<decltype(p)>> T;
    for (size_t i = 0; i < n; ++i)
      for (int turn = 1; p[i] == (T)~(T)0; ++turn) {
        if (turn % 64 == 0 && std::chrono::steady_clock::now() - t0 > kAwaitAtMost) return false;
        __builtin_ia32_pause();
      }
    return true;
  };
  for (const Awaited& a : awaited_) {
    if (a.size == 4 ? arrived((volatile uint32_t*)a.at, a.elements) : arrived((volatile uint16_t*)a.at, a.elements)) continue;
    net_->Wait();  // a long pass, or outputs that hold that value: then it is of no use here
    settled_ = true;
    passes_unsettled_ = 0;
    const uint8_t* bytes = (const uint8_t*)a.at;
    for (size_t i = 0; i < a.elements; ++i) {
      uint32_t v = 0;
      memcpy(&v, bytes + i * a.size, a.size);
      if (v == (a.size == 4 ? 0xffffffffu : 0xffffu)) await_outputs_ = false;
    }
    break;
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  return true;
}

// Whether each operator's results reach an output: only then is a pass whose outputs have arrived done with all its memory.
bool Predictor::EveryOperatorFeedsAnOutput() const {
  std::vector<Blob*> needed = external_output_blob_;
  const auto& ops = net_->GetOperators();
  for (auto it = ops.rbegin(); it != ops.rend(); ++it) {
    if ((*it)->type() == "ConstantFill") continue;  // (the net's, or nobody's any more where operators were folded)
    const auto& out = (*it)->Outputs();
    const bool used = std::any_of(out.begin(), out.end(), [&](Blob* b) { return std::find(needed.begin(), needed.end(), b) != needed.end(); });
    if (!used) return false;
    needed.insert(needed.end(), (*it)->Inputs().begin(), (*it)->Inputs().end());
  }
  return true;
}

// what is queued on ctx's stream from here on runs behind the last pass
void Predictor::SettleBefore(const HIPContext& ctx) {
  if (!settled_ && ctx.stream_serial() != forward_on_) Settle();
}

// the last pass has ended on the device as well
void Predictor::Settle() {
  if (settled_) return;
  for (Blob* b : external_output_blob_) {
    if (b->device_type() != kHIP) continue;
    HIPContext ctx(b->device_option());
    ctx.Activate();
    HIP_CHECK(ctx.stream_serial() == forward_on_ ? hipStreamSynchronize(ctx.hip_stream()) : WaitForDevice());
    break;
  }
  settled_ = true;
  passes_unsettled_ = 0;
}

void Predictor::WithdrawHostCopies() {
  for (size_t i = 0; i < external_output_blob_.size(); ++i)
    if (output_sole_[i]) external_output_blob_[i]->host_copy() = Blob::HostCopy();
}

void Predictor::QueueOutputs() {
  hipStream_t st = (hipStream_t)net_->WaitedStream();
  bz_feed_rows rows[BZ_FEED_MAX_ROWS];
  size_t which[BZ_FEED_MAX_ROWS];
  int n = 0;
  for (size_t i = 0; i < external_output_blob_.size(); ++i) {
    Blob* blob = external_output_blob_[i];
    const size_t bytes = blob->size() * DataTypeSize(blob->data_type());
    const bool ahead = st != nullptr && CopiedAhead(i) && blob->pitch() == 0 && blob->data() != nullptr && bytes > 0 &&
                       bytes <= std::min(kCopiedAheadMax, HostHalf(i));
    output_wanted_[i] = false;
    if (ahead && output_sole_[i] && blob->host_copy().copied == bytes) {
      output_ahead_[i] = output_by_operator_[i] = true;
      if (Awaitable(i)) awaited_.push_back({blob->host_copy().at, blob->size(), DataTypeSize(blob->data_type())});
    } else if (ahead && n < BZ_FEED_MAX_ROWS) {
      rows[n].src = blob->data();
      rows[n].dst = (char*)output_cpu_[i]->data() + (1 - output_half_[i]) * HostHalf(i);
      rows[n].rows = 1;
      rows[n].row_bytes = rows[n].src_pitch = rows[n].dst_pitch = (int64_t)bytes;
      if (Awaitable(i)) {
        memset(rows[n].dst, kNotThereByte, bytes);
        awaited_.push_back({rows[n].dst, blob->size(), DataTypeSize(blob->data_type())});
      }
      which[n++] = i;
    }
  }
  if (n == 0) return;
  if (bz_feed(nullptr, nullptr, 0, rows, n, st) != 0) {  // (not launched: Output copies by itself)
    awaited_.clear();
    return;
  }
  for (int k = 0; k < n; ++k) output_ahead_[which[k]] = true;
}

bool Predictor::Output(const char* name, void** data, size_t* len) {
  const int idx = OutputName2Idx(name);
  if (idx < 0) {
    LOG_ERROR("The name: %s is not The output of net", name);
    return false;
  }
  return Output((size_t)idx, data, len);
}
bool Predictor::Output(size_t idx, void** data, size_t* len) {
  if (idx >= external_output_blob_.size()) {
    LOG_ERROR("The idx=%zu exceed size=%zu", idx, external_output_blob_.size());
    return false;
  }
  Blob* blob = external_output_blob_[idx];
  if (blob->unplaced()) {
    LOG_ERROR("output %s is an input that was reshaped beyond its fed size and has not been fed since", net_->external_output()[idx].c_str());
    return false;
  }
  const size_t bytes = blob->size() * DataTypeSize(blob->data_type());
  try {
    if (blob->device_type() == kCPU) {
      *data = blob->data();
    } else {
      Blob* cpu = output_cpu_[idx].get();
      output_wanted_[idx] = true;
      if (output_ahead_[idx]) {  // (a second Output of the same pass copies again)
        output_half_[idx] = 1 - output_half_[idx];
        output_ahead_[idx] = false;
      } else {
        cpu->set_data_type((DataType)blob->data_type());
        const bool two = bytes <= kCopiedAheadMax;
        cpu->Reshape({two ? 2 * ((blob->size() + kHalfAlign - 1) / kHalfAlign * kHalfAlign) : blob->size()});
        output_pinned_[idx] = IsPinnedHost(cpu->data());
        if (HostHalf(idx) < bytes) output_half_[idx] = 0;
        Settle();
        HIPContext ctx(blob->device_option());
        ctx.Activate();
        CopyBytes((char*)cpu->data() + output_half_[idx] * HostHalf(idx), kCPU, blob->data(), kHIP, bytes, ctx.hip_stream());
      }
      output_read_[idx] = bytes;
      *data = (char*)cpu->data() + output_half_[idx] * HostHalf(idx);
    }
  } catch (std::exception& e) {
    LOG_ERROR("output failed: %s", e.what());
    return false;
  }
  if (len) *len = bytes;
  return true;
}

const std::vector<size_t>& Predictor::OutputShape(size_t idx) const {
  BLAZE_CONDITION_THROW(idx < external_output_blob_.size(), "The idx=", idx, " blob is null");
  return external_output_blob_[idx]->shape();
}
const std::vector<size_t>& Predictor::OutputShape(const char* name) const {
  const int idx = OutputName2Idx(name);
  BLAZE_CONDITION_THROW(idx >= 0, "The name ", name, " is not Output of net");
  return OutputShape((size_t)idx);
}
int Predictor::OutputDataType(const char* name) const {
  const int idx = OutputName2Idx(name);
  return idx < 0 ? (int)kPDT_Invalid : external_output_blob_[idx]->data_type();
}

std::vector<std::string> Predictor::ListInternalName() const {
  std::vector<std::string> names;
  for (const auto& it : net_->workspace()->constant_blobs()) names.push_back(it.first);
  return names;
}
bool Predictor::InternalParam(const char* name, void** data, size_t* len) {
  const auto& m = net_->workspace()->constant_blobs();
  auto it = m.find(name);
  if (it == m.end()) return false;
  Blob* blob = it->second;
  const size_t bytes = blob->size() * DataTypeSize(blob->data_type());
  try {
    if (blob->device_type() == kCPU) {
      *data = blob->data();
    } else {
      DeviceOption cpu_opt;
      cpu_opt.set_device_type(kCPU);
      auto& cpu = param_cpu_[name];
      if (!cpu) cpu = std::make_shared<Blob>(cpu_opt);
      cpu->set_data_type((DataType)blob->data_type());
      cpu->Reshape(blob->shape());
      HIPContext ctx(blob->device_option());
      ctx.Activate();
      CopyBytes(cpu->data(), kCPU, blob->data(), kHIP, bytes, ctx.hip_stream());
      *data = cpu->data();
    }
  } catch (std::exception& e) {
    LOG_ERROR("param copy failed: %s", e.what());
    return false;
  }
  if (len) *len = bytes;
  return true;
}
const std::vector<size_t>& Predictor::InternalShape(const char* name) const {
  const auto& m = net_->workspace()->constant_blobs();
  auto it = m.find(name);
  BLAZE_CONDITION_THROW(it != m.end(), "The name ", name, " is not a parameter of net");
  return it->second->shape();
}
int Predictor::InternalDataType(const char* name) const {
  const auto& m = net_->workspace()->constant_blobs();
  auto it = m.find(name);
  return it == m.end() ? (int)kPDT_Invalid : it->second->data_type();
}

void Predictor::RegisterObservers(const std::vector<std::string>& names) {
  for (const auto& n : names)
    if (n == "profile") net_->set_profile(true);
}
void Predictor::DumpObservers(std::unordered_map<std::string, std::string>* dump_map) {
  (*dump_map)["profile"] = net_->DumpProfile();
  std::stringstream ss;
  ss << "{";
  for (size_t i = 0; i < output_ahead_.size(); ++i)
    ss << (i ? "," : "") << "\"" << net_->external_output()[i] << "\":\"" << (!output_ahead_[i] ? "device" : output_by_operator_[i] ? "operator" : "copied") << "\"";
  ss << "}";
  (*dump_map)["outputs"] = ss.str();
  (*dump_map)["pass"] = settled_ ? "ended" : "arrived";
}

void* Predictor::InputDevicePtr(const char* name) {
  const int idx = InputName2Idx(name);
  if (idx >= 0 && external_input_blob_[idx]->unplaced()) {  // outgrew its feed-arena slice: memory of its own
    Blob* blob = external_input_blob_[idx];
    const std::vector<TIndex> shape = blob->shape();
    blob->DropArenaView();
    blob->Reshape(shape);
  }
  // (a strided input -- one that lives inside a Concat's output -- has no plain buffer to hand out)
  return idx < 0 || external_input_blob_[idx]->pitch() != 0 ? nullptr : HandOut(external_input_blob_[idx]);
}
void* Predictor::OutputDevicePtr(const char* name) {
  const int idx = OutputName2Idx(name);
  return idx < 0 ? nullptr : HandOut(external_output_blob_[idx]);
}
void* Predictor::HandOut(Blob* blob) {
  Settle();
  output_ahead_.assign(output_ahead_.size(), false);
  if (std::find(handed_out_.begin(), handed_out_.end(), blob) == handed_out_.end()) handed_out_.push_back(blob);
  return blob->data();
}

std::string& last_error_for_thread() {
  static thread_local std::string s;
  return s;
}

// ------------------------------------------------------------------------------------------ manager
std::shared_ptr<store::SparsePuller>& PredictorManager::EnsureSparsePuller(const char* type) {
  if (!sparse_puller_) sparse_puller_.reset(store::SparsePullerCreationRegisterer::Get()->CreateSparsePuller(type));
  return sparse_puller_;
}

bool PredictorManager::LoadSparseModelWeight(const char* uri, const char* type) {
  try {
    sparse_puller_.reset(store::SparsePullerCreationRegisterer::Get()->CreateSparsePuller(type));
    if (store::kOK != sparse_puller_->Load(uri)) {
      LOG_ERROR("load sparse model %s failed", uri);
      return false;
    }
  } catch (std::exception& e) {
    LOG_ERROR("load sparse model %s failed: %s", uri, e.what());
    last_error_for_thread() = e.what();
    return false;
  }
  return true;
}

bool PredictorManager::LoadModel(const char* filename, bool optimization_pass) {
  return LoadModel(filename, "", kBlaze, optimization_pass);
}
bool PredictorManager::LoadDeepNetModel(const char* model_conf, const char* model_data, bool optimization_pass) {
  return LoadModel(model_conf, model_data, kUlf, optimization_pass);
}
bool PredictorManager::LoadModel(const char* conf_file, const char*, ModelType model_type, bool) {
  if (model_type != kBlaze) {
    LOG_ERROR("model type %d needs an importer that is not part of this build; convert the model to a Blaze NetDef first", model_type);
    last_error_for_thread() = "unsupported model type";
    return false;
  }
  std::string err;
  NetDef def;
  if (!LoadNetDefFromFile(conf_file, &def, &err)) {
    LOG_ERROR("Load model %s failed: %s", conf_file, err.c_str());
    last_error_for_thread() = err;
    return false;
  }
  return LoadNetDef(def);
}
bool PredictorManager::LoadNetDef(const NetDef& net_def) {
  std::lock_guard<std::mutex> lock(mutex_);
  net_def_ = net_def;
  if (!run_mode_.empty()) net_def_.run_mode_ = run_mode_;
  has_net_ = true;
  workspace_.clear();
  return true;
}

Predictor* PredictorManager::CreatePredictor(PredictDeviceType predict_device, int device_id) {
  std::lock_guard<std::mutex> lock(mutex_);
  try {
    BLAZE_CONDITION_THROW(has_net_, "no model loaded");
    if (device_id < 0) device_id = 0;
    DeviceOption device_option;
    switch (predict_device) {
      case kPDT_CPU:
        device_option.set_device_type(kCPU);
        device_option.set_device_id(0);
        break;
      case kPDT_HIP:
        device_option.set_device_type(kHIP);
        device_option.set_device_id(device_id);
        break;
      default: {  // ProbeDevice (predictor_manager_impl.cc:162-177): round robin over the visible accelerators
        static int next = 0;
        int count = 0;
        HIP_CHECK(hipGetDeviceCount(&count));
        BLAZE_CONDITION_THROW(count > 0, "no accelerator visible and this build has no CPU path");
        device_option.set_device_type(kHIP);
        device_option.set_device_id(next++ % count);
      }
    }
    const int dt = device_option.device_type(), di = device_option.device_id();
    auto& ws = workspace_[dt][di];
    if (!ws) {
      ws.reset(new Workspace());
      ws->Init(net_def_);
      auto* opt = ws->net_def()->mutable_device_option();
      opt->set_device_type(dt);
      opt->set_device_id(di);
      // the device of the predictor overrides what individual operators were exported with
      for (auto& op : ws->net_def()->op_) {
        if (op.has_device_option()) {
          op.device_option_.set_device_type(dt);
          op.device_option_.set_device_id(di);
        }
      }
      ws->SetSparsePuller(sparse_puller_);
    }
    std::shared_ptr<Net> net = ws->CreateNet();
    BLAZE_CONDITION_THROW(net != nullptr, "net creation failed");
    return new Predictor(net);
  } catch (std::exception& e) {
    LOG_ERROR("Create Model Predictor failed, msg=%s", e.what());
    last_error_for_thread() = e.what();
    return nullptr;
  }
}

bool InitScheduler(bool, int, int, int, int, int) { return true; }

}  // namespace blaze
