// Pinned words that a kernel leaves its results in: checks, and the use on a stream
// that keeps the host allocator from giving the memory to others before the kernel is
// through (as a non-blocking copy's would be).
#pragma once

#include <ATen/hip/CachingHostAllocator.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/extension.h>

inline long* pinned_words(const c10::optional<at::Tensor>& host, long n) {
  if (!host.has_value()) return nullptr;
  TORCH_CHECK(host->is_pinned() && host->scalar_type() == at::kLong &&
                  host->is_contiguous() && host->numel() >= n,
              "host must be pinned words, one a row");
  at::getHostAllocator(at::kCUDA)->record_event(
      host->data_ptr(), host->storage().data_ptr().get_context(),
      c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().unwrap());
  return host->data_ptr<long>();
}
