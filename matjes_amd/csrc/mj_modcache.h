// Modules compiled in this process, by device and source: a module is loaded on
// one device, and its functions run there only.  The objects that run a module's
// functions hold it; the store holds the `keep` last asked for beside them, so
// that a later object with the same source finds it, and a module that neither
// holds is unloaded (by the module type's destructor).  Plain C++ (the module
// type is a parameter), so that the host test compiles it by itself.
#pragma once
#include <stddef.h>

#include <list>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <utility>

template <class Mod>
class ModCache {
  public:
    using Ref = std::shared_ptr<Mod>;
    explicit ModCache(size_t keep) : keep_(keep) {}

    // the module of a source on a device: make(ref) compiles and loads it there
    // unless it is kept (nonzero: failed, nothing kept)
    template <class Make>
    int get(int device, const std::string &src, Ref *out, Make make)
    {
        Ref old;   // unloaded, if at all, after the lock is gone
        std::lock_guard<std::mutex> lk(mu_);
        auto it = at_.find({device, src});
        if (it != at_.end()) {
            last_.splice(last_.begin(), last_, it->second);
        } else {
            Ref m;
            if (int rc = make(&m)) return rc;
            ++made_;
            it = at_.emplace(std::make_pair(device, src), last_.end()).first;
            last_.push_front({it, std::move(m)});
            it->second = last_.begin();
        }
        *out = last_.front().mod;
        if (last_.size() > keep_) {
            old = std::move(last_.back().mod);
            at_.erase(last_.back().key);
            last_.pop_back();
        }
        return 0;
    }

    // modules made so far, and kept now
    void stats(long long *made, long long *kept)
    {
        std::lock_guard<std::mutex> lk(mu_);
        *made = made_;
        *kept = (long long)last_.size();
    }

  private:
    struct Entry;
    using List = std::list<Entry>;
    using Map = std::map<std::pair<int, std::string>, typename List::iterator>;
    struct Entry {
        typename Map::iterator key;
        Ref mod;
    };
    const size_t keep_;
    long long made_ = 0;
    std::mutex mu_;
    List last_;   // the last asked for first
    Map at_;
};
