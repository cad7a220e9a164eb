// bd_cpus.h -- how many CPUs this process may keep busy.
#pragma once

#include <sched.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <string>

namespace bd {

// The two numbers of a CPU quota, period of which quota may be used: from one
// file ("quota period", cgroup v2), or from two (v1).  "max" or -1 is no quota.
// Whole CPUs, at least one; none when there is no quota.
inline int whole_cpus(long long quota, long long period, int none) {
    if (quota <= 0 || period <= 0) return none;
    return (int)std::max(1LL, std::min<long long>(quota / period, none));
}

inline bool read_line(const std::string &path, char *line, int size) {
    FILE *f = fopen(path.c_str(), "r");
    if (!f) return false;
    const bool ok = fgets(line, size, f) != nullptr;
    fclose(f);
    return ok;
}

// CPUs that the CPU quotas of this process's control groups leave it, of n:
// groups is /proc/self/cgroup, tree /sys/fs/cgroup.  A group's own quota and
// those of the groups above it all hold; a container mostly sees its own group
// as the root.
inline int quota_cpus(int n, const std::string &groups, const std::string &tree) {
    FILE *f = fopen(groups.c_str(), "r");
    if (!f) return n;
    int least = n;
    char line[4096], text[128];
    while (fgets(line, sizeof(line), f)) {  // id:controllers:/path
        line[strcspn(line, "\n")] = 0;
        char *names = strchr(line, ':');
        char *path = names ? strchr(names + 1, ':') : nullptr;
        if (!path) continue;
        *path++ = 0;
        ++names;
        const bool v2 = !*names;
        bool cpu = v2;
        for (char *s = names, *save = nullptr; (s = strtok_r(s, ",", &save)); s = nullptr)
            cpu = cpu || !strcmp(s, "cpu");
        if (!cpu) continue;
        for (std::string at = path;;) {
            const std::string dir = tree + (v2 ? "" : "/cpu") + (at == "/" ? "" : at);
            long long quota = 0, period = 0;
            if (v2) {
                if (read_line(dir + "/cpu.max", text, sizeof(text)) &&
                    sscanf(text, "%lld %lld", &quota, &period) == 2)
                    least = std::min(least, whole_cpus(quota, period, n));
            } else if (read_line(dir + "/cpu.cfs_quota_us", text, sizeof(text)) &&
                       sscanf(text, "%lld", &quota) == 1 &&
                       read_line(dir + "/cpu.cfs_period_us", text, sizeof(text)) &&
                       sscanf(text, "%lld", &period) == 1) {
                least = std::min(least, whole_cpus(quota, period, n));
            }
            const size_t cut = at.rfind('/');
            if (cut == std::string::npos || at == "/" || at.empty()) break;
            at = cut == 0 ? "/" : at.substr(0, cut);
        }
    }
    fclose(f);
    return least;
}

inline int affinity_cpus() {
    cpu_set_t set;
    return sched_getaffinity(0, sizeof(set), &set) == 0 ? std::max(1, CPU_COUNT(&set)) : 1;
}

// CPUs of the affinity mask, and no more than the quotas leave.
inline int usable_cpus() {
    return quota_cpus(affinity_cpus(), "/proc/self/cgroup", "/sys/fs/cgroup");
}

}  // namespace bd
