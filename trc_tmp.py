import sys, json, torch
from perf import cases
c = json.loads(sys.argv[1])
n = int(sys.argv[2]) if len(sys.argv) > 2 else 25
s = cases.prepare(c, 1)
for _ in range(n): cases.run(s)
torch.cuda.synchronize()
