// Which assemblies of a context are recorded as a HIP graph and replayed. Host only.
#pragma once

namespace fem2d {

// what a recorded assembly depends on besides its buffers
struct GraphKey {
  unsigned long long domain = 0;
  int basis = -1, ai = -1, bi = -1, nu = 0, nv = 0;
  long long capacity = -1;
  unsigned long long alloc_generation = 0;
  bool run_large = true;  // the block path's launches are part of it
  int precision = -1;
  int chunk = 0;
  bool operator==(const GraphKey& o) const {
    return domain == o.domain && basis == o.basis && ai == o.ai && bi == o.bi && nu == o.nu && nv == o.nv &&
           capacity == o.capacity && alloc_generation == o.alloc_generation && run_large == o.run_large &&
           precision == o.precision && chunk == o.chunk;
  }
};

// An assembly is recorded the second time in a row that its key comes, and replayed
// while the key stays. One that is not repeated is launched kernel by kernel: a Domain
// of an adaptive loop or of a drop-in call is assembled only once, and a recording
// costs more than the launches it saves (the assembly of a new hp-irregular 32 x 16
// Domain 310 us recorded and replayed, 177 launched).
class GraphRule {
 public:
  enum Step { kLaunch, kRecord, kReplay };
  Step step(const GraphKey& key) const {
    return key == recorded_ ? kReplay : key == latest_ ? kRecord : kLaunch;
  }
  // the graph of the recorded key is about to be destroyed / the graph of key was made
  void forget() { recorded_ = GraphKey{}; }
  void made(const GraphKey& key) { recorded_ = key; }
  // key's assembly was launched, recorded or replayed
  void came(const GraphKey& key) { latest_ = key; }
  // whether it had row groups of the block path. A Domain's first assembly runs that
  // path's kernels whether or not they have work, and the ones that follow only if they do:
  // its key is kept as the next one will have it.
  void learned(bool large) { latest_.run_large = large; }

 private:
  GraphKey recorded_, latest_;
};

}  // namespace fem2d
