// Modules compiled in this process, by device and source: a module is loaded on
// one device, and its functions run there only.  Plain C++ (the module type is
// a parameter), so that the host test compiles it by itself.
#pragma once
#include <map>
#include <mutex>
#include <string>
#include <utility>

template <class Mod>
class ModCache {
  public:
    // the module of a source on a device: make(mod) compiles and loads it there on
    // first use (nonzero: failed, nothing kept)
    template <class Make>
    int get(int device, const std::string &src, Mod *out, Make make)
    {
        std::lock_guard<std::mutex> lk(mu_);
        auto it = mods_.find({device, src});
        if (it == mods_.end()) {
            Mod m{};
            if (int rc = make(&m)) return rc;
            it = mods_.emplace(std::make_pair(device, src), m).first;
        }
        *out = it->second;
        return 0;
    }

  private:
    std::mutex mu_;
    std::map<std::pair<int, std::string>, Mod> mods_;
};
