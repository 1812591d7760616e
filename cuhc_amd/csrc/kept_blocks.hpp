// Freed blocks kept for the next request of the same key (size class, or device
// and size), the oldest given up first where a new one would pass the limit: a
// process that goes through many sizes keeps those of its latest calls. (With
// the new block given up instead, stale sizes held the limit and every large
// request mapped its pages anew: 14.4 GB took 330 ms per call.)
// No lock and no HIP types: the owner has both.
#pragma once

#include <stddef.h>

#include <iterator>
#include <list>
#include <map>
#include <new>
#include <vector>

namespace cuhc {

template <class Key> class KeptBlocks {
public:
  // The block of this key put last, or null.
  void *take(const Key &key) {
    const auto it = byKey_.find(key);
    if (it == byKey_.end())
      return nullptr;
    const auto block = it->second.back();
    it->second.pop_back();
    if (it->second.empty())
      byKey_.erase(it);
    void *p = block->p;
    bytes_ -= block->bytes;
    order_.erase(block);
    return p;
  }

  // Whether the block is kept; release(p) is called for what makes way.
  template <class Release>
  bool put(const Key &key, void *p, size_t bytes, size_t limit, Release &&release) {
    if (bytes > limit)
      return false;
    while (bytes_ > limit - bytes)
      release(oldest());
    try {
      order_.push_back(Block{key, p, bytes});
    } catch (const std::bad_alloc &) {
      return false;
    }
    try {
      byKey_[key].push_back(std::prev(order_.end()));
    } catch (const std::bad_alloc &) {
      const auto it = byKey_.find(key);
      if (it != byKey_.end() && it->second.empty())
        byKey_.erase(it);
      order_.pop_back();
      return false;
    }
    bytes_ += bytes;
    return true;
  }

  template <class Release> void clear(Release &&release) {
    while (!order_.empty())
      release(oldest());
  }

  size_t bytes() const { return bytes_; }

private:
  struct Block {
    Key key;
    void *p;
    size_t bytes;
  };

  // Takes out the oldest block: the first of its key, as blocks of a key are put
  // at the back and taken from there.
  void *oldest() {
    const Block block = order_.front();
    const auto it = byKey_.find(block.key);
    it->second.erase(it->second.begin());
    if (it->second.empty())
      byKey_.erase(it);
    order_.pop_front();
    bytes_ -= block.bytes;
    return block.p;
  }

  std::list<Block> order_; // oldest first
  std::map<Key, std::vector<typename std::list<Block>::iterator>> byKey_;
  size_t bytes_ = 0;
};

} // namespace cuhc
